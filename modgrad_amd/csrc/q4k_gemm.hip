// Prefill dequant-GEMM on the gfx950 matrix cores:
//   C[m][r] = sum_k dequant(W)[r][k] * A[m][k],  A f16 [M][K], C f32 [M][N].
// No counterpart in the reference (its prefill is a per-token GEMV loop,
// crates/modgrad-gemma/examples/gemma4_rocm.rs:26-34); each weight is the
// canonical dequantized value (gguf.rs:364-404) times a power of two 2^(e-20)
// that keeps it inside f16's normal range, with d*sc and dmin*m (times their
// powers of two) rounded to f16 and the weight computed and rounded once in
// f16; C is scaled back exactly.
//
// One kernel, gemm_q4k_f16_kernel, in tile shapes from 32 rows x 16 tokens to
// 336 x 128 (kTiles), picked per call by a model of the time of each
// (gemm_f16_launch).
//
// Work-group = NWK groups of wavefronts, each with its own share of the
// K blocks (b = kg, kg + NWK, ...): NWN compute wavefronts along W's rows and
// one loader wavefront.
//   * A compute wavefront owns 16 RT rows and all 16 TT tokens of the tile
//     (RT x TT v_mfma_f32_16x16x32_f16 tiles, W rows the A operand, tokens
//     the B operand, so a lane's 4 accumulators are 4 consecutive rows of one
//     token: one 16-byte store into C). It loads its rows' 16-byte qs pieces
//     straight into registers PD blocks ahead, and dequantizes them there:
//     every weight is dequantized once per tile, and W never goes through
//     LDS.
//   * The loader copies the tokens' 128-value half blocks from memory
//     straight into LDS (global_load_lds, no registers): NBUF half blocks
//     before the first product, then NBUF - 1 ahead. It issues no other
//     vector memory operation, so its vmcnt waits are exact (a register
//     spilled around them would make them stricter); the compute wavefronts'
//     loads are waited for by the compiler.
//   * The two wavefronts of a SIMD run a half block's dequantization and
//     products in opposite orders (run), so that one's vector work falls under
//     the other's matrix work: 3584 x 18944 at 512 tokens 105 -> 95 us, at 4096
//     553 -> 508.
//   * One barrier per half block. After the K loop the NWK partial tiles are
//     added in LDS in a fixed order (the result does not depend on timing).
// Splitting K inside the work-group is what fills the chip when there are few
// rows (o and down: 3584) or few tokens: with 128-row tiles over all of K,
// 3584 x 18944 had 28 work-groups per 128 tokens for 256 CUs.
//
// k order. Lane (row l = lane % 16, q = lane / 16) holds qs bytes
// 16 q .. 16 q + 15 of half block H (qs bytes 64 H ..). MFMA slot (j, hi) of
// the half takes its bytes 8 j .. 8 j + 7, low or high nibbles: the lane
// group's k are 64 (q / 2) + 16 (q % 2) + 8 j + 32 hi + 0..7 of the half, so
// the token operand is one 16-byte chunk, number 8 (q / 2) + 2 (q % 2) + j +
// 4 hi, of the token's half block. A token's 16 chunks sit in LDS at
// chunk ^ (token % 16): the reads have no bank conflicts (counted: 0), and
// the loader applies the swizzle to the addresses it reads from.
//
// Dequantization. A nibble in bits 4..7 of an f16 is the subnormal q * 2^-20,
// exact (low nibbles are shifted there, a dword at a time); one v_pk_fma_f16
// with the sub-block pair (d*sc*2^e, -dmin*m*2^(e-20)) gives two weights *
// 2^(e-20), rounded once: 2.75 VALU per pair with the byte permutes (low
// nibbles left in bits 0..3 would save a shift per eight weights and cost four
// binades of the weights' range). Each lane decodes one row's block header (a
// row on four lanes, a quarter each, when RT == 1) into 8 such pairs in a
// wave-private LDS table, one block ahead.
//
// Range. Each W row carries a running power-of-two exponent e. A block's
// `tight` is the largest e that keeps its 63|d| * 2^e and 63|dmin| * 2^(e-19)
// below 2^16, so that neither the multipliers nor the weights pass f16's
// maximum. A row keeps e while tight - 2 kRangeHeadroom <= e <= tight; a block
// outside that (the first nonzero one always is) sets e to its
// tight - kRangeHeadroom, up or down, and the wavefront multiplies its sums so
// far by 2^(e_new - e_old) (exact) before that block's products. A block's
// largest multiplier is then 2^9 .. 2^16 and its d*sc*q * 2^(e-20) reach
// 2^-8 .. 2^0: every sub-block, 2^6 below its block's largest or not, is held
// in normal f16 numbers but for what a block's largest weights round away.
// Sums in f32 do not overflow: a weight is below 2^15 in its own e, an
// activation below 2^16, and e (-10 .. 53 over all finite headers) rises by 63
// at most. C is multiplied by 2^(20-e) at the end.
#include "q4k_device.hpp"
#include "q4k_launch.hpp"

namespace mgq {

namespace gemm {
constexpr int NXCD = 8;             // XCDs the hardware deals work-groups across, round robin
constexpr int kRangeHeadroom = 3;   // blocks 2^3 either way of the first: no rescale
constexpr int kNoExp = 100;         // e of a row with no nonzero block yet (tight <= 53)
constexpr int SROW = 40;            // bytes per scale-table row (32 + pad: conflict-free b64 reads)
constexpr int GROUP_M = 8;          // token tiles that share an XCD's W tiles
}  // namespace gemm

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

// Two weights from the quants 16 q in two bytes of v (pick: v_perm selector)
// as an f16 pair.
__device__ __forceinline__ uint32_t dqs2(uint32_t v, uint32_t pick, h2_t d1, h2_t nm1) {
    const h2_t q = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(v, v, pick));
    return __builtin_bit_cast(uint32_t, q * d1 + nm1);
}

// Byte B of v as a float (written out: the compiler, knowing that the byte has
// six bits, takes two operations).
template <int B>
__device__ __forceinline__ float ubyte_f32(uint32_t v) {
    float f;
    if constexpr (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 3) asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(v));
    return f;
}
// half_bits_finite in one operation less.
__device__ __forceinline__ float finite_half(uint32_t h) {
    const float f = (float)__builtin_bit_cast(_Float16, (uint16_t)h);
    return fabsf(f) < 65536.0f ? f : 0.0f;  // infinities and NaN -> 0
}

// Copies 16 bytes per lane from base + off to LDS bytes dst + 16 * lane (no
// registers; the compiler sets M0). The caller waits with vm_wait.
template <class Off>
__device__ __forceinline__ void lds_copy16(uint8_t *dst, const uint8_t *base, Off &off) {
    asm("" : "+s"(base));  // base and offset kept apart: no address arithmetic per copy
    asm("" : "+v"(off));
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(base + off),
                                     (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
// At most N of this wavefront's vector memory operations still in flight.
template <int N>
__device__ __forceinline__ void vm_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
}
// Work-group barrier behind this wavefront's LDS operations; unlike
// __syncthreads it leaves global loads and copies in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int RT, int TT, int NWN, int NWK, int NBUF>
struct GemmLayout {
    static constexpr int BN = 16 * RT * NWN, BM = 16 * TT;  // rows, tokens of a tile
    static constexpr int NC = NWN * NWK;                    // compute wavefronts
    static constexpr int NT = 64 * (NC + NWK);
    static constexpr int IPS = BM / 4;                      // copies (4 tokens x 256 B) per half block
    static constexpr uint32_t SA = BM * 256;                // one half block of the tokens
    static constexpr uint32_t ST = RT * 16 * gemm::SROW;    // one scale table of a wavefront
    static constexpr uint32_t OS = NWK * NBUF * SA;
    static constexpr uint32_t MAIN = OS + NC * 2 * ST;
    static constexpr uint32_t RED = (NWK - 1) * NWN * RT * TT * 1024;  // partial tiles, over the rest
    static constexpr uint32_t LDS = MAIN > RED ? MAIN : RED;
    static_assert(LDS <= 160 * 1024, "LDS of one CU");
};

// Off: unsigned type of byte offsets inside a tile (uint32_t unless the rows
// are so long that a tile spans 4 GiB).
template <int RT, int TT, int NWN, int NWK, int NBUF, int PD, class Off>
__global__ __launch_bounds__(64 * (NWN + 1) * NWK) void gemm_q4k_f16_kernel(
    const uint8_t *__restrict__ w, const uint16_t *__restrict__ a, float *__restrict__ c, int n,
    int bpr, int m_tokens, int tiles_n, int tiles_m) {
    using L = GemmLayout<RT, TT, NWN, NWK, NBUF>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    // work-group -> tile: work-group i runs on XCD i % 8; XCD x takes a
    // contiguous range of tiles. Tiles go in bands of GROUP_M token tiles,
    // token tiles fastest, so an XCD's work-groups share W and A lines in its
    // L2.
    const int ntiles = tiles_n * tiles_m;
    const int per_xcd = (ntiles + gemm::NXCD - 1) / gemm::NXCD;
    const int tile = (int)(blockIdx.x % gemm::NXCD) * per_xcd + (int)(blockIdx.x / gemm::NXCD);
    if (tile >= ntiles) return;  // uniform; only when ntiles % 8 != 0
    const int band = tile / (gemm::GROUP_M * tiles_n), in_band = tile - band * gemm::GROUP_M * tiles_n;
    const int band_m = min(gemm::GROUP_M, tiles_m - band * gemm::GROUP_M);
    const int n0 = (in_band / band_m) * L::BN, m0 = (band * gemm::GROUP_M + in_band % band_m) * L::BM;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int NB = (bpr + NWK - 1) / NWK;  // blocks per K share (the last may be past the end)
    auto blk = [&](int b) __attribute__((always_inline)) { return min(b, bpr - 1); };

    if (wave >= L::NC) {
        // ---- loader of K share kg: half block s & 1 of block kg + (s / 2) NWK
        // goes to buffer s % NBUF. Copy i moves tokens 4i .. 4i + 3; lane
        // (token 4i + lane / 16) fetches the chunk that belongs at its place.
        // Tokens past m_tokens re-read the last one (never stored).
        const int kg = wave - L::NC;
        const uint32_t buf0 = (uint32_t)kg * NBUF * L::SA;
        const size_t pitch = (size_t)bpr * kBlockElems * 2;
        const uint8_t *abase = reinterpret_cast<const uint8_t *>(a) + (size_t)m0 * pitch;
        Off aoff[L::IPS];
#pragma unroll
        for (int i = 0; i < L::IPS; ++i) {
            const int t = 4 * i + q;
            aoff[i] = (Off)min(t, m_tokens - 1 - m0) * (Off)pitch + 16u * (l16 ^ (t & 15));
        }
        auto half_at = [&](int s) __attribute__((always_inline)) {
            return abase + (size_t)blk(kg + (s >> 1) * NWK) * (kBlockElems * 2) + 256 * (s & 1);
        };
        auto buf_at = [&](int s) __attribute__((always_inline)) { return buf0 + (uint32_t)(s % NBUF) * L::SA; };
        if (((uintptr_t)a & 15u) == 0) {
            auto copy = [&](int s) __attribute__((always_inline)) {
                const uint8_t *src = half_at(s);
                uint8_t *dst = lds + buf_at(s);
#pragma unroll
                for (int i = 0; i < L::IPS; ++i) lds_copy16(dst + 1024u * i, src, aoff[i]);
            };
#pragma unroll
            for (int s = 0; s < NBUF; ++s) copy(s);
            vm_wait<(NBUF - 1) * L::IPS>();  // half block 0 has landed
            lds_barrier();
            for (int s = 0; s < 2 * NB; ++s) {
                vm_wait<(NBUF - 2) * L::IPS>();  // half block s + 1 has landed
                lds_barrier();                   // half block s has been read
                copy(s + NBUF);
            }
            vm_wait<0>();
        } else {
            // A off 16 bytes: through registers, half block s in set s % D, D
            // half blocks in flight (18944 x 3584 at 512 tokens: 321 us with
            // two pieces in flight -> 78, aligned 78-82)
            constexpr int D = L::IPS <= 8 ? 4 : L::IPS <= 16 ? 2 : 1;
            u32x4 R[D][L::IPS];
            auto fetch = [&](int s, int set) __attribute__((always_inline)) {
                const uint8_t *src = half_at(s);
#pragma unroll
                for (int i = 0; i < L::IPS; ++i) {
                    asm("" : "+v"(aoff[i]));  // not widened to a register pair
                    R[set][i] = ld_u32x4(src + aoff[i]);
                }
            };
            auto put = [&](int s, int set) __attribute__((always_inline)) {
                uint8_t *dst = lds + buf_at(s) + 16 * lane;
#pragma unroll
                for (int i = 0; i < L::IPS; ++i) *reinterpret_cast<u32x4 *>(dst + 1024u * i) = R[set][i];
                __builtin_amdgcn_sched_barrier(0);  // the set's next loads take its registers
            };
#pragma unroll
            for (int s = 0; s < D; ++s) fetch(s, s);
            put(0, 0);
            fetch(D, 0);
            lds_barrier();
            for (int s0 = 0; s0 < 2 * NB; s0 += D) {
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    const int s = s0 + u;
                    if (s >= 2 * NB) break;  // uniform
                    // into the buffer of half block s + 1 - NBUF, read before
                    // the barrier that half block s began behind
                    put(s + 1, (u + 1) % D);
                    fetch(s + 1 + D, (u + 1) % D);
                    lds_barrier();  // half block s has been read
                }
            }
        }
        if constexpr (NWK > 1) {  // the partial tiles' two barriers
            lds_barrier();
            lds_barrier();
        }
        return;
    }

    const int wn = wave % NWN, kg = wave / NWN;
    const size_t row_bytes = (size_t)bpr * kBlockBytes;
    // this wavefront's rows r0 ..; rows past n re-read the last row
    const int r0 = n0 + wn * 16 * RT, rb = min(r0, n - 1);
    const uint8_t *wbase = w + (size_t)rb * row_bytes;
    Off woff[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
        woff[i] = (Off)(min(r0 + 16 * i + l16, n - 1) - rb) * (Off)row_bytes + 16u * q;
    // header loads: a row a lane, 64 rows a load (RT == 1, 2: a row on 4, 2 lanes)
    constexpr int HD = (RT + 3) / 4;
    Off hoff[HD];
#pragma unroll
    for (int k = 0; k < HD; ++k) {
        const int row = RT == 1 ? l16 : RT == 2 ? (lane & 31) : min(64 * k + lane, 16 * RT - 1);
        hoff[k] = (Off)(min(r0 + row, n - 1) - rb) * (Off)row_bytes;
    }
    u32x4 Wr[PD][2][RT], Hd[PD][HD];  // qs and headers of the next PD blocks
    auto loadW = [&](int b, auto hc, auto uc) __attribute__((always_inline)) {
        constexpr int H = decltype(hc)::value, U = decltype(uc)::value;
        const uint8_t *p = wbase + (size_t)blk(b) * kBlockBytes;
#pragma unroll
        for (int i = 0; i < RT; ++i) Wr[U][H][i] = ld_u32x4(p + woff[i] + 16 + 64 * H);
    };
    auto loadH = [&](int b, auto uc) __attribute__((always_inline)) {
        const uint8_t *p = wbase + (size_t)blk(b) * kBlockBytes;
#pragma unroll
        for (int k = 0; k < HD; ++k) Hd[decltype(uc)::value][k] = ld_u32x4(p + hoff[k]);
    };
    // ---- block headers -> scale table `buf`; true when some row's e changed
    // (its sums so far then take a factor 2^del). No branches: a header decodes
    // in the shadow of the products around it. `on` is false past the end of
    // the K share.
    int er[HD], del[HD];
#pragma unroll
    for (int k = 0; k < HD; ++k) { er[k] = gemm::kNoExp; del[k] = 0; }
    uint8_t *stab = lds + L::OS + wave * (2 * L::ST);
    // (RT <= 2: the lane's sub-blocks are in the first or the second half)
    const bool first4 = q < 2;
    const uint32_t mA = first4 ? 0x3F3F3F3Fu : 0x0F0F0F0Fu, mB = first4 ? 0u : 0x30303030u, qsh = 16u * (q & 1);
    // the sub-block pair in bytes B, B + 1 of sc and mn (even one, odd one)
    auto pairs = [](float d, float nm, uint32_t sc, uint32_t mn, auto bc) __attribute__((always_inline)) {
        constexpr int B = decltype(bc)::value;
        const h2_t lo = {(_Float16)(d * ubyte_f32<B>(sc)), (_Float16)(nm * ubyte_f32<B>(mn))};
        const h2_t hi = {(_Float16)(d * ubyte_f32<B + 1>(sc)), (_Float16)(nm * ubyte_f32<B + 1>(mn))};
        return u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
    };
    using B0 = std::integral_constant<int, 0>;
    using B2 = std::integral_constant<int, 2>;
    auto decode = [&](auto uc, int buf, bool on) __attribute__((always_inline)) -> bool {
        constexpr int U = decltype(uc)::value;
        bool any = false;
#pragma unroll
        for (int k = 0; k < HD; ++k) {
            const uint32_t h0 = Hd[U][k][0], s0 = Hd[U][k][1], s1 = Hd[U][k][2], s2 = Hd[U][k][3];
            const float dh = finite_half(h0), mh = finite_half(h0 >> 16);
            // 15 - exponent of the bound (a normal number, or zero; 64.1: f16
            // rounds below 65504)
            const float bound = fabsf(dh) * 64.1f + fabsf(mh) * (63.0f / 524288.0f);
            const int tight = 15 + 127 - (int)(__builtin_bit_cast(uint32_t, bound) >> 23);
            const bool out = on && bound > 0.0f && (uint32_t)(tight - er[k]) > 2 * gemm::kRangeHeadroom;
            const int e = out ? tight - gemm::kRangeHeadroom : er[k];
            del[k] = e - er[k];
            any |= out;
            er[k] = e;
            const float d = ldexpf(dh, e), nm = -ldexpf(mh, e - 20);
            if constexpr (RT <= 2) {
                const uint32_t sc = ((first4 ? s0 : s2) & mA) | ((s0 >> 2) & mB);
                const uint32_t mn = ((first4 ? s1 : s2 >> 4) & mA) | ((s1 >> 2) & mB);
                if constexpr (RT == 1) {  // lane group q: sub-blocks 2q, 2q + 1
                    *reinterpret_cast<u32x2 *>(stab + buf * L::ST + l16 * gemm::SROW + 8 * q) = pairs(d, nm, sc >> qsh, mn >> qsh, B0{});
                } else {  // half-wavefront h: sub-blocks 4h .. 4h + 3
                    u32x2 *dst = reinterpret_cast<u32x2 *>(stab + buf * L::ST + (lane & 31) * gemm::SROW + 16 * (lane >> 5));
                    dst[0] = pairs(d, nm, sc, mn, B0{});
                    dst[1] = pairs(d, nm, sc, mn, B2{});
                }
            } else {
                const int row = min(64 * k + lane, 16 * RT - 1);
                u32x2 *dst = reinterpret_cast<u32x2 *>(stab + buf * L::ST + row * gemm::SROW);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t sc = scales4(j, s0, s2), mn = mins4(j, s1, s2);
                    dst[2 * j] = pairs(d, nm, sc, mn, B0{});
                    dst[2 * j + 1] = pairs(d, nm, sc, mn, B2{});
                }
            }
        }
        return __any(any);
    };
    // 2^x of row 16 i + 4 q + v, x from the lane that decodes the row
    auto row_pow2 = [&](const int(&x)[HD], int i, int add, int sign) __attribute__((always_inline)) {
        f32x4 f;
#pragma unroll
        for (int v = 0; v < 4; ++v) f[v] = ldexpf(1.0f, add + sign * __shfl(x[i / 4], 16 * (i % 4) + 4 * q + v, 64));
        return f;
    };

    f32x4 acc[RT][TT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t chunk0 = (uint32_t)(8 * (q >> 1) + 2 * (q & 1));
    const uint8_t *abuf0 = lds + (uint32_t)kg * NBUF * L::SA + l16 * 256;
    u32x4 op[RT][4];  // W operands of a half block: slot (j, hi) at 2 hi + j
    u32x2 sp[RT];
    auto read_scales = [&](int H, int tab) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
            sp[i] = *reinterpret_cast<const u32x2 *>(stab + tab * L::ST + (16 * i + l16) * gemm::SROW + 16 * H + 8 * (q >> 1));
    };
    auto dequant = [&](auto hc, auto uc) __attribute__((always_inline)) {
        constexpr int H = decltype(hc)::value, U = decltype(uc)::value;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const uint32_t sp0 = sp[i][0], sp1 = sp[i][1];
            const h2_t sl = __builtin_bit_cast(h2_t, sp0), sh = __builtin_bit_cast(h2_t, sp1);
            const h2_t dl = {sl[0], sl[0]}, nl = {sl[1], sl[1]}, dh = {sh[0], sh[0]}, nh = {sh[1], sh[1]};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t v = Wr[U][H][i][u], lo = (v << 4) & 0xF0F0F0F0u, hi = v & 0xF0F0F0F0u;
                constexpr uint32_t B01 = 0x0C010C00u, B23 = 0x0C030C02u;  // bytes -> 0, 2
                op[i][u >> 1][2 * (u & 1)] = dqs2(lo, B01, dl, nl);
                op[i][u >> 1][2 * (u & 1) + 1] = dqs2(lo, B23, dl, nl);
                op[i][2 + (u >> 1)][2 * (u & 1)] = dqs2(hi, B01, dh, nh);
                op[i][2 + (u >> 1)][2 * (u & 1) + 1] = dqs2(hi, B23, dh, nh);
            }
        }
    };
    // The late order's half 1 operands are made where dequant stands and not
    // sunk behind the barrier into the products' branch, where they would stand
    // in the early order, beside the SIMD's other wavefront, and hold their
    // half block's registers past the next loads, which then need a copy and a
    // wait at the end of every block. (With half 0's
    // pinned too, 224 x 128 gains 2 % and the 160-row tiles lose 1-3 %.)
    auto pin = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(op[i][s]));
    };
    constexpr int SETS = TT <= 3 ? 4 : 2;  // slots whose token operands are in registers
    half8 tb[SETS][TT];
    auto read = [&](int s, int buf) __attribute__((always_inline)) {
        const uint8_t *p = abuf0 + buf * L::SA + ((chunk0 + (s & 1) + 4 * (s >> 1)) ^ (uint32_t)l16) * 16;
#pragma unroll
        for (int j = 0; j < TT; ++j) tb[s % SETS][j] = *reinterpret_cast<const half8 *>(p + j * 4096);
    };
    auto read_ahead = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < (SETS == 4 ? 4 : 1); ++s) read(s, buf);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if constexpr (SETS == 2) {
                if (s < 3) read(s + 1, buf);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < TT; ++j)
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, op[i][s]),
                                                                        tb[s % SETS][j], acc[i][j], 0, 0, 0);
        }
    };

    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    int buf = 0;
    auto next_buf = [&]() __attribute__((always_inline)) {
        lds_barrier();
        buf = buf + 1 == NBUF ? 0 : buf + 1;
    };
    auto rescale = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const f32x4 f = row_pow2(del, i, 0, 1);
#pragma unroll
            for (int j = 0; j < TT; ++j) acc[i][j] *= f;
        }
    };
    // Two orders of the same work, one for the even and one for the odd
    // wavefronts of each SIMD, so that one dequantizes while the other
    // multiplies: (late = 0) a half block's dequantization, then its products;
    // (late = 1) its products, then the next half block's dequantization. The
    // next block's header is decoded in half 1 or half 0. Loads go out in one
    // order, the prologue's included, so that every wait leaves the younger
    // ones in flight.
    auto run = [&](auto late) __attribute__((always_inline)) {
        constexpr bool LATE = decltype(late)::value;
        loadH(kg, H0{});
        __builtin_amdgcn_sched_barrier(0);
        decode(H0{}, 0, NWK == 1 || kg < bpr);
        auto first = [&](auto uc) __attribute__((always_inline)) {
            constexpr int U = decltype(uc)::value;
            if constexpr (U < PD) {
                loadW(kg + U * NWK, H0{}, uc);
                __builtin_amdgcn_sched_barrier(0);
                loadH(kg + (U + 1) * NWK, std::integral_constant<int, (U + 1) % PD>{});
                __builtin_amdgcn_sched_barrier(0);
                loadW(kg + U * NWK, H1{}, uc);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        first(H0{});
        first(H1{});
        if constexpr (LATE) {
            asm volatile("" ::: "memory");  // other lanes' table entries: read after decode's stores
            read_scales(0, 0);
            dequant(H0{}, H0{});
            __builtin_amdgcn_sched_barrier(0);
            loadW(kg + PD * NWK, H0{}, H0{});
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();  // half block 0 is in LDS
        auto block = [&](int t, auto uc) __attribute__((always_inline)) {
            constexpr int U = decltype(uc)::value;
            using N = std::integral_constant<int, (U + 1) % PD>;  // the next block's registers
            const int b = kg + t * NWK, tab = t & 1;
            const bool live = NWK == 1 || b < bpr;  // uniform
            const bool on = NWK == 1 || b + NWK < bpr;
            bool changed = false;
            if constexpr (LATE) {
                if (live) {
                    read_ahead(buf);
                    products(buf);
                }
                read_scales(1, tab);
                changed = decode(N{}, tab ^ 1, on);
                __builtin_amdgcn_sched_barrier(0);
                loadH(b + (1 + PD) * NWK, N{});
                dequant(H1{}, uc);
                pin();
                __builtin_amdgcn_sched_barrier(0);
                loadW(b + PD * NWK, H1{}, uc);
                __builtin_amdgcn_sched_barrier(0);
                next_buf();
                if (live) {
                    read_ahead(buf);
                    products(buf);
                }
                read_scales(0, tab ^ 1);
                dequant(H0{}, N{});
                __builtin_amdgcn_sched_barrier(0);
                loadW(b + (1 + PD) * NWK, H0{}, N{});
                __builtin_amdgcn_sched_barrier(0);
            } else {
                if (live) {
                    read_scales(0, tab);
                    read_ahead(buf);
                    dequant(H0{}, uc);
                    products(buf);
                }
                __builtin_amdgcn_sched_barrier(0);
                loadW(b + PD * NWK, H0{}, uc);
                __builtin_amdgcn_sched_barrier(0);
                next_buf();
                changed = decode(N{}, tab ^ 1, on);
                __builtin_amdgcn_sched_barrier(0);
                loadH(b + (1 + PD) * NWK, N{});
                if (live) {
                    read_scales(1, tab);
                    read_ahead(buf);
                    dequant(H1{}, uc);
                    products(buf);
                }
                __builtin_amdgcn_sched_barrier(0);
                loadW(b + PD * NWK, H1{}, uc);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (changed) rescale();  // rare
            next_buf();
        };
        static_assert(PD == 1 || PD == 2, "blocks of W in registers");
        for (int t = 0; t < NB; t += PD) {
            block(t, H0{});
            if constexpr (PD == 2)
                if (t + 1 < NB) block(t + 1, H1{});
        }
    };
    // (336 x 128's accumulators leave no registers for the second order)
    constexpr bool PAIRED = L::NC > 4 && RT * TT <= 16;
    if (PAIRED && (wave & 4)) run(std::integral_constant<bool, PAIRED>{});
    else run(std::false_type{});
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const f32x4 f = row_pow2(er, i, 20, -1);
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] *= f;
    }

    if constexpr (NWK > 1) {
        // shares 1 .. hand their tiles over in LDS (lane-linear, over the
        // token buffers); share 0 adds them in order and stores
        lds_barrier();  // every wavefront, the loaders' copies included, is done with them
        f32x4 *red = reinterpret_cast<f32x4 *>(lds) + lane;
        auto at = [&](int g, int i, int j) { return ((((g - 1) * NWN + wn) * RT + i) * TT + j) * 64; };
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < TT; ++j) red[at(kg, i, j)] = acc[i][j];
        }
        lds_barrier();
        if (kg > 0) return;
        for (int g = 1; g < NWK; ++g)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < TT; ++j) acc[i][j] += red[at(g, i, j)];
    }

    // lane: rows r0 + 16 i + 4 q + v of token m0 + 16 j + l16
    const bool vec = (n % 4) == 0 && (((uintptr_t)c & 15u) == 0);
#pragma unroll
    for (int j = 0; j < TT; ++j) {
        const int m = m0 + 16 * j + l16;
        if (m >= m_tokens) continue;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int r = r0 + 16 * i + 4 * q;
            float *dst = c + (size_t)m * n + r;
            if (vec && r + 3 < n) {
                *reinterpret_cast<f32x4 *>(dst) = acc[i][j];
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (r + v < n) dst[v] = acc[i][j][v];
            }
        }
    }
}

template <int RT, int TT, int NWN, int NWK, int NBUF, int PD, class Off>
static hipError_t launch_tile(const uint8_t *w, const uint16_t *a, float *c, int n, int bpr, int m_tokens,
                              hipStream_t stream) {
    using L = GemmLayout<RT, TT, NWN, NWK, NBUF>;
    auto kern = gemm_q4k_f16_kernel<RT, TT, NWN, NWK, NBUF, PD, Off>;
    static std::atomic<int> lds_state[64];  // one per instance: no lock on a launch
    const hipError_t attr = allow_full_lds((const void *)kern, lds_state);
    if (attr != hipSuccess || w == nullptr) return attr;  // w null: attribute only (gemm_prepare)
    const int tn = (n + L::BN - 1) / L::BN, tm = (m_tokens + L::BM - 1) / L::BM;
    const long ntiles = (long)tn * tm;
    const long grid = (ntiles + gemm::NXCD - 1) / gemm::NXCD * gemm::NXCD;
    if (grid > 0x7FFFFFFFL) return hipErrorInvalidValue;
    kern<<<(unsigned)grid, L::NT, L::LDS, stream>>>(w, a, c, n, bpr, m_tokens, tn, tm);
    return hipGetLastError();
}

// The tile shapes. A work-group of one takes fixed_us + block_us per block of
// its K share, with every CU holding one; a call takes as many rounds of that
// as its tiles fill (rounds of all CUs, the last one counted whole). The times
// rank the shapes, they do not predict a call: large calls take 13-17 %
// longer. Fitted to 438 shapes (N 576-37888, K 1536-18944, M 17-2048), 32 x 16
// again on 700 others (N 33-47104, K 1536-26624, M 1-4096): over these the
// picked shape is within 0.1 % of the best one on average, 7 % at worst.
// W's prefetch is two blocks where that was faster; 32 x 32 and 32 x 48 would
// hold two without losing a wavefront, and the same to 1 % with them.
struct GemmTile {
    int bn, bm, nwk;
    float fixed_us, block_us;
    hipError_t (*launch)(const uint8_t *, const uint16_t *, float *, int, int, int, hipStream_t);
};
#define MGQ_TILE(RT, TT, NWN, NWK, NBUF, PD, FIXED, BLOCK) \
    {16 * RT * NWN, 16 * TT, NWK, FIXED, BLOCK, launch_tile<RT, TT, NWN, NWK, NBUF, PD, uint32_t>}
static const GemmTile kTiles[] = {
    MGQ_TILE(1, 1, 2, 4, 4, 2, 2.2f, 1.12f),   //  32 x  16
    MGQ_TILE(1, 2, 2, 4, 4, 1, 2.2f, 1.43f),   //  32 x  32
    MGQ_TILE(1, 3, 2, 4, 3, 1, 2.4f, 1.68f),   //  32 x  48
    MGQ_TILE(1, 3, 4, 2, 3, 2, 2.7f, 1.31f),   //  64 x  48
    MGQ_TILE(2, 5, 2, 2, 3, 2, 3.8f, 1.48f),   //  64 x  80
    MGQ_TILE(2, 3, 4, 2, 4, 1, 3.7f, 1.92f),   // 128 x  48
    MGQ_TILE(2, 4, 4, 2, 3, 1, 4.3f, 2.11f),   // 128 x  64
    MGQ_TILE(2, 5, 4, 2, 3, 1, 5.1f, 2.32f),   // 128 x  80
    MGQ_TILE(1, 3, 10, 1, 4, 2, 3.8f, 1.30f),  // 160 x  48
    MGQ_TILE(2, 3, 5, 2, 4, 1, 4.4f, 2.31f),   // 160 x  48, K in two shares
    MGQ_TILE(2, 5, 5, 2, 3, 1, 5.9f, 2.77f),   // 160 x  80
    MGQ_TILE(2, 8, 7, 1, 2, 1, 6.4f, 2.80f),   // 224 x 128
    MGQ_TILE(3, 5, 7, 1, 3, 1, 6.0f, 2.70f),   // 336 x  80
    MGQ_TILE(3, 8, 7, 1, 2, 1, 7.7f, 3.69f),   // 336 x 128
};
#undef MGQ_TILE
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
// Rows so long that the offsets inside any tile pass 32 bits (K above 2^27).
static constexpr auto launch_wide = launch_tile<1, 2, 2, 4, 4, 1, uint64_t>;

hipError_t gemm_prepare() {
    hipError_t e = launch_wide(nullptr, nullptr, nullptr, 0, 0, 0, nullptr);
    for (const GemmTile &t : kTiles)
        if (e == hipSuccess) e = t.launch(nullptr, nullptr, nullptr, 0, 0, 0, nullptr);
    return e;
}

// The shape of a call: an index of kTiles, or kNumTiles for launch_wide.
static int gemm_pick(int n, int bpr, int m_tokens, long cus) {
    int best = kNumTiles;
    float best_us = 0.0f;
    for (int i = 0; i < kNumTiles; ++i) {
        const GemmTile &t = kTiles[i];
        // offsets of a tile's rows and tokens are 32-bit
        if ((int64_t)t.bn * bpr * kBlockBytes > 0xFFFFFFFFll || (int64_t)t.bm * bpr * kBlockElems * 2 > 0xFFFFFFFFll)
            continue;
        const long tiles = (long)((n + t.bn - 1) / t.bn) * ((m_tokens + t.bm - 1) / t.bm);
        const float us = (float)((tiles + cus - 1) / cus) * (t.fixed_us + t.block_us * (float)((bpr + t.nwk - 1) / t.nwk));
        if (best == kNumTiles || us < best_us) {
            best = i;
            best_us = us;
        }
    }
    return best;
}

int gemm_tile_shape(int n, int bpr, int m_tokens, int cus, int *rows, int *tokens, int *k_shares) {
    const int i = gemm_pick(n, bpr, m_tokens, cus);
    *rows = i < kNumTiles ? kTiles[i].bn : 32;
    *tokens = i < kNumTiles ? kTiles[i].bm : 32;
    *k_shares = i < kNumTiles ? kTiles[i].nwk : 4;
    return i;
}

hipError_t gemm_f16_launch(const uint8_t *w, const uint16_t *a, float *c, int n, int bpr,
                           int m_tokens, hipStream_t stream) {
    if ((uintptr_t)a & 1u) return hipErrorInvalidValue;
    const int i = gemm_pick(n, bpr, m_tokens, device_cus());
    return (i < kNumTiles ? kTiles[i].launch : launch_wide)(w, a, c, n, bpr, m_tokens, stream);
}

}  // namespace mgq
