// qs_logits.hip - the output layer alone: logits[r][v] = sum_k H[r][k] W[v][k], bf16 operands
// and fp32 accumulation on the matrix cores (forward_cpu.c:319-323 at bf16), for up to 256
// rows against the weights packed by k_head_pack.
//
// What bounds it: W (2 V E bytes) is read from HBM once and the logits (4 V rows) are written
// once; at 256 rows x 2048 x 151,936 that is 622 + 156 MB against 159 GFLOP, so the layer
// streams.  W reaches the CUs at (bytes in flight) / (load latency), the CUs have to stream
// until the end, and what the products cost beside the stream shows.  Hence:
//
//   * One workgroup of 8 wavefronts per CU with nearly all of its 160 KB of LDS: a ring of
//     H stages (from the XCD's L2, short latency) and a ring of W stages (HBM) of 20 KB.
//     Loads return in order per wavefront, so the two rings belong to different wavefronts:
//     0-3 load H, 4-7 load W, each waits for its own, and the stage's barrier joins them.  60
//     to 120 KB of W are in flight a CU; one 128-column tile a workgroup, two of them a CU
//     with three shared stages (qs_head.hip's shape), held 32.
//   * The vocabulary is dealt out in 32-column blocks, an equal run for each workgroup (18 or
//     19 blocks at V = 151,936 on 256 CUs).  Tiles of 128 columns made 1,187 workgroups for
//     512 places: a third round with two thirds of the chip idle.
//   * A run is cut into tiles of at most 10 blocks (H is staged again for each: 0.5 GB through
//     L2 at 256 rows, against 1.2 GB for tiles of 128 columns; 8 blocks: 210 us against 192
//     at this point of the work) whose stages follow each other in the rings without a break:
//     while a tile's accumulators are stored, the next tile's loads are in flight.  The
//     stores go straight from the accumulators (32 lanes, 128 consecutive bytes a row).
//   * A stage issues a fixed number of loads whose addresses are one scalar offset away from
//     the last stage's (buffer loads; what lies outside reads nothing), so a stage costs no
//     address arithmetic and no branches: 192 -> 170 us.
//
// Measured, the layer alone in bursts, before (qs_head.hip's kernels) -> now: 256 rows x 2048
// x 151,936 240 -> 170 us (4.6 TB/s), 128 rows 165 -> 129, 64 rows 138 -> 114, 32 rows 122 ->
// 105, 1 row 108 -> 93 (6.7 TB/s); 256 x 4096 x 75,968 262 -> 157.  Two halves of the
// wavefronts alternating reads and products behind four barriers a stage: 231.
//
// One stage is 32 embedding elements; the sums run over k in steps of 16 in ascending order,
// the order of qs_head.hip's fused kernels, so both write the same logits.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/quasar_sampler.h"
#include "qs_device.h"
#include "qs_internal.h"
#include "qs_launch.h"

namespace {

constexpr int LT = QS_HEAD_TILE;        // columns per packed tile
constexpr int LK = 32;                  // embedding elements per stage
constexpr int LNT = 512;                // threads: 8 wavefronts

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct LinArgs {
    const uint16_t *h;                  // [n_rows][E] bf16 bits
    const uint16_t *w;                  // packed weights (k_head_pack), bf16 bits
    int E, n_rows, V, nblk;             // nblk: 32-column blocks of the vocabulary
    float *logits;                      // [n_rows][V]
};

// The shape for up to RB rows: RG row groups of WRB 32-row blocks x CG column groups (the
// wavefronts) of a tile of at most TB 32-column blocks; HS and WS ring slots.
template <int RB> struct LinShape;
template <> struct LinShape<256> { static constexpr int WRB = 2, RG = 4, CG = 2, TB = 10, HS = 3, WS = 5; };
template <> struct LinShape<128> { static constexpr int WRB = 2, RG = 2, CG = 4, TB = 10, HS = 4, WS = 6; };
template <> struct LinShape<64> { static constexpr int WRB = 2, RG = 1, CG = 8, TB = 10, HS = 5, WS = 7; };
template <> struct LinShape<32> { static constexpr int WRB = 1, RG = 1, CG = 8, TB = 10, HS = 5, WS = 7; };

// 64 bytes a row or column, its four 16-byte segments stored in the order
// seg ^ ((row / 4) % 4): the lanes of an operand read hit distinct banks.
template <int RB>
struct LinLds {
    uint16_t h[LinShape<RB>::HS][RB < 64 ? 64 : RB][LK];   // (4 wavefronts x 16 rows at least)
    uint16_t w[LinShape<RB>::WS][LinShape<RB>::TB * 32][LK];
};
static_assert(sizeof(LinLds<256>) <= 160 * 1024 && sizeof(LinLds<128>) <= 160 * 1024 &&
                  sizeof(LinLds<64>) <= 160 * 1024, "one workgroup's LDS");

// Wait until at most N of this wavefront's vector memory operations are in flight.
template <int N>
__device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N <= 63, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A barrier without __syncthreads()'s fence, which would wait for every load in flight; the
// wavefront's LDS reads are done before it.
__device__ __forceinline__ void lin_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// NT: W by nontemporal loads.
template <int RB, bool NT>
__device__ __forceinline__ void lin_run(const LinArgs &a) {
    using S = LinShape<RB>;
    constexpr int WRB = S::WRB, RG = S::RG, CG = S::CG, TB = S::TB, HS = S::HS, WS = S::WS;
    constexpr int NB = (TB + CG - 1) / CG;          // a wavefront's blocks at most
    constexpr int WL = TB / 2;                      // W pieces a wavefront 4..7 loads at most
    static_assert(RG * CG == 8 && RG * WRB * 32 == RB && TB % 2 == 0 && WL <= 5 && NB <= 5, "the wavefronts");
    constexpr int HPIECES = RB / 16;                // 1 KB pieces of an H stage
    constexpr int HL = (HPIECES + 3) / 4;           // of them a wavefront 0..3 loads
    __shared__ __attribute__((aligned(16))) LinLds<RB> L;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = a.n_rows, E = a.E, V = a.V;
    const int nst = E / LK;
    const int b0 = (int)((int64_t)a.nblk * blockIdx.x / gridDim.x);
    const int b1 = (int)((int64_t)a.nblk * (blockIdx.x + 1) / gridDim.x);
    const int nbk = b1 - b0, ntile = (nbk + TB - 1) / TB;
    if (nbk <= 0) return;
    // tile t of the run: blocks [tile_begin(t), tile_begin(t + 1))
    const int per = nbk / ntile, extra = nbk - per * ntile;
    auto tile_begin = [&](int t) { return b0 + per * t + min(t, extra); };

    const bool wload = wv >= 4;                     // this wavefront loads W (else H)
    // The load side: the next stage's tile and stage within it, its ring slot, and each piece's
    // byte offset in the wavefront's operand.  Every stage issues the same number of loads, so
    // the waits are constants: pieces past the tile's columns or the batch's rows, and all of
    // them past the run's last stage, lie past the operand's buffer and read no memory.  W's
    // buffer is the packed tiles of this run, its base formed in 64 bits: W as a whole may pass
    // the 4 GiB that a buffer's size and offsets hold (256,000 x 12,288 is 6.3 GB), a run does
    // not (qs_logits_fits).
    constexpr int NL = WL > HL ? WL : HL;
    constexpr uint32_t NONE = 0xFFFFFFF0u;
    const int t0 = b0 * 32 / LT, t1 = (b1 * 32 + LT - 1) / LT;      // the run's packed tiles
    const uint16_t *wrun = a.w + (int64_t)t0 * E * LT;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        wload ? (void *)wrun : (void *)a.h, 0,
        (int)(wload ? (uint32_t)(t1 - t0) * (uint32_t)E * (2 * LT) : (uint32_t)B * (uint32_t)E * 2u),
        0x00020000);                                // raw buffer, 32-bit data format
    int lt = 0, ls = 0, lslot = 0;
    uint32_t off[NL];
    auto load_tile = [&]() {
        const int tb = tile_begin(lt), nb = lt < ntile ? tile_begin(lt + 1) - tb : 0;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int p = (wv & 3) + 4 * i;
            if (wload) {                            // 16 columns, 1 KB, already swizzled
                const int col = tb * 32 + p * 16;
                off[i] = p < 2 * nb ? ((uint32_t)(col / LT - t0) * (uint32_t)(nst * 8) +
                                       (uint32_t)(col % LT / 16)) * 1024u + (uint32_t)lane * 16u
                                    : NONE;
            } else {                                // rows 16 p .. + 16
                const int r = p * 16 + (lane >> 2);
                off[i] = r < B && p < HPIECES && lt < ntile
                             ? 2u * ((uint32_t)r * (uint32_t)E +
                                     (uint32_t)(((lane & 3) ^ ((r >> 2) & 3)) * 8))
                             : NONE;
            }
        }
    };
    load_tile();
    auto issue = [&]() __attribute__((always_inline)) {
        if (wload) {
            uint16_t *dst = &L.w[lslot][(wv & 3) * 16][0];
            const int at = ls * (LT * LK * 2);
#pragma unroll
            for (int i = 0; i < WL; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(dst + i * 64 * LK), 16,
                                                         (int)off[i], at, 0, NT ? 2 : 0);
            lslot = lslot + 1 == WS ? 0 : lslot + 1;
        } else {
            uint16_t *dst = &L.h[lslot][(wv & 3) * 16][0];
            const int at = ls * (LK * 2);
#pragma unroll
            for (int i = 0; i < HL; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(dst + i * 64 * LK), 16,
                                                         (int)off[i], at, 0, 0);
            lslot = lslot + 1 == HS ? 0 : lslot + 1;
        }
        if (++ls == nst) {
            ls = 0;
            ++lt;
            load_tile();
        }
    };
    for (int g = 0; g < (wload ? WS : HS) - 1; ++g) issue();

    // wavefront w: rows 32 WRB (w % RG) .. + 32 WRB; blocks w / RG + CG j of a tile
    const int rg = wv % RG, cg = wv / RG;
    const int rr = lane & 31, swz = (rr >> 2) & 3;
    int hslot = 0, wslot = 0;
    auto tile = [&](auto nbc, int tb) __attribute__((always_inline)) {
        constexpr int NBW = decltype(nbc)::value;   // this wavefront's blocks
        f32x16 acc[WRB][NBW > 0 ? NBW : 1];
#pragma unroll
        for (int i = 0; i < WRB; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j) acc[i][j] = f32x16{};
        u32x4 ha[2][WRB], wb[2][NBW > 0 ? NBW : 1];
        auto read = [&](int ks) __attribute__((always_inline)) {
            const int sg = ((ks * 2 + (lane >> 5)) ^ swz) * 8;
            if constexpr (NBW > 0) {
#pragma unroll
                for (int i = 0; i < WRB; ++i)
                    ha[ks][i] = *(const u32x4 *)&L.h[hslot][(rg * WRB + i) * 32 + rr][sg];
#pragma unroll
                for (int j = 0; j < NBW; ++j)
                    wb[ks][j] = *(const u32x4 *)&L.w[wslot][(cg + CG * j) * 32 + rr][sg];
            }
        };
        auto multiply = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int i = 0; i < WRB; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, ha[ks][i]), __builtin_bit_cast(bf16x8, wb[ks][j]),
                        acc[i][j], 0, 0, 0);
        };
        for (int st = 0; st < nst; ++st) {
            // this stage's own loads are in (the later stages' stay in flight; stores of an
            // earlier tile among them only make the wait longer)
            if (wload) vm_wait<(WS - 2) * WL>();
            else vm_wait<(HS - 2) * HL>();
            // the slots refilled next were read before this barrier by every wavefront
            lin_barrier();
            read(0);
            read(1);
            issue();
            multiply(0);
            multiply(1);
            hslot = hslot + 1 == HS ? 0 : hslot + 1;
            wslot = wslot + 1 == WS ? 0 : wslot + 1;
        }
        int r0 = rg * WRB * 32 + (lane >> 5) * 4;
        asm volatile("" : "+v"(r0));                // (its row addresses are formed here, not
                                                    // held through the products)
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const int col = (tb + cg + CG * j) * 32 + rr;
            float *out = a.logits + (int64_t)r0 * V + col;
#pragma unroll
            for (int i = 0; i < WRB; ++i) {
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int dr = i * 32 + (q >> 2) * 8 + (q & 3);
                    if (r0 + dr < B && col < V) out[(int64_t)dr * V] = acc[i][j][q];
                }
            }
        }
    };
    for (int t = 0; t < ntile; ++t) {
        const int tb = tile_begin(t), nb = tile_begin(t + 1) - tb;
        const int mine = nb > cg ? (nb - cg + CG - 1) / CG : 0;   // (uniform)
        if constexpr (NB >= 5)
            if (mine == 5) tile(std::integral_constant<int, 5>{}, tb);
        if constexpr (NB >= 4)
            if (mine == 4) tile(std::integral_constant<int, 4>{}, tb);
        if constexpr (NB >= 3)
            if (mine == 3) tile(std::integral_constant<int, 3>{}, tb);
        if constexpr (NB >= 2)
            if (mine == 2) tile(std::integral_constant<int, 2>{}, tb);
        if (mine == 1) tile(std::integral_constant<int, 1>{}, tb);
        if (mine == 0) tile(std::integral_constant<int, 0>{}, tb);
    }
    vm_wait<0>();                                   // nothing may land in the LDS after the end
}

// One kernel per shape (a template kernel's host stub is not emitted here).
#define LIN_KERNEL(RB)                                                                        \
    __global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))         \
    k_logits##RB(LinArgs a) { lin_run<RB, false>(a); }                                        \
    __global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))         \
    k_logits##RB##_nt(LinArgs a) { lin_run<RB, true>(a); }
LIN_KERNEL(32)
LIN_KERNEL(64)
LIN_KERNEL(128)
LIN_KERNEL(256)
#undef LIN_KERNEL

// W is read nontemporally where it and the logits together pass the last-level cache (256 MB):
// there W would only push out the logits, which the pick reads next (16 rows x 2048: 51.6
// against 58.0 us at 328 MB of weights, 64 rows: 113.6 against 131.8 at 622 MB; 256 rows x 512
// x 151,936, 156 + 156 MB: 70 against 72).  What fits stays in it from one step to the next
// (128 rows x 512 x 151,936, 156 + 78 MB: 41.5 against 46.8 us; 256 x 1024 x 80,000, 164 + 82
// MB: 58 against 64; at 205 + 3 MB the two are even).
constexpr uint64_t NT_BYTES = 256ull << 20;
uint64_t layer_bytes(int n_embd, int n_rows, int n_vocab) {
    return (2ull * (uint64_t)n_embd + 4ull * (uint64_t)n_rows) * (uint64_t)n_vocab;
}

}  // namespace

// Microseconds, the tile kernels / this file's, W from HBM (matrices in turn past the last-level
// cache) unless said otherwise:
//   * up to one 128-column tile a CU there is nothing to balance (V = 32,000: 1 row x 512 6.6 /
//     7.4, 40 rows x 4096 43 / 45, 256 x 4096 91 / 100);
//   * a short run is all ramp: E = 64, 1 row 4.0 / 4.8 at V = 32,772, 7.0 / 8.0 at 128,256; 64
//     rows x 256 11.5 / 12.3 at 64,000, 23.3 / 24.8 at 151,936.  128 rows x 256 13.7 / 10.9 at
//     32,772, 33.1 / 31.7 at 151,936; 64 rows x 512 15.2 / 12.5 and 38.2 / 36.8;
//   * up to 64 rows that do not pass the last-level cache, the tiles (two a CU at once) lose
//     only in a round that is not full: 1 row x 512 at 1,002 tiles of 1,024 places (V = 128,256)
//     24.9 / 27.1, in the cache 21.4 / 22.1, at 500 of 512 (64,000) 14.4 / 14.5 and 12.2 / 13.4;
//     at 782 of 1,024 (100,000) 22.6 / 20.9 and 19.1 / 18.2, at 257 of 512 11.5 / 10.4.
// Past it: 1 row x 2048 x 128,256 89 / 81, 64 rows x 2048 x 100,000 100 / 78 (128,256 x 1536 is
// the exception: 68 / 77 at 1 row, 111 / 107 at 128).
bool qs_logits_pays(int n_embd, int n_rows, int n_vocab, int n_cu) {
    const int tiles = (n_vocab + LT - 1) / LT, places = 2 * n_cu;
    if (tiles <= n_cu || n_embd < 256) return false;
    if (n_rows > 64 || layer_bytes(n_embd, n_rows, n_vocab) > NT_BYTES) return true;
    const int rounds = (tiles + places - 1) / places;
    return n_embd >= 512 && 20 * (int64_t)tiles < 19 * (int64_t)rounds * places;
}

bool qs_logits_fits(int n_embd, int n_rows, int n_vocab, int n_cu) {
    // (a run of ceil(blocks / n_cu) blocks of 32 columns touches at most this many tiles)
    const int64_t blocks = ((n_vocab + 31) / 32 + n_cu - 1) / n_cu;
    const int64_t run = (blocks * 32 + LT - 1) / LT + 1;
    const int64_t w = run * n_embd * (2 * LT), h = (int64_t)n_rows * n_embd * 2;
    return w < 0xFFFFFFF0ll && h < 0xFFFFFFF0ll;
}

int qs_logits_launch(const void *d_hidden, const void *d_weight, int n_embd, int n_rows,
                     int n_vocab, float *d_logits, int n_cu, hipStream_t stream) {
    LinArgs a;
    a.h = (const uint16_t *)d_hidden;
    a.w = (const uint16_t *)d_weight;
    a.E = n_embd;
    a.n_rows = n_rows;
    a.V = n_vocab;
    a.nblk = (n_vocab + 31) / 32;
    a.logits = d_logits;
    const unsigned grid = (unsigned)n_cu;             // (n_vocab > 128 n_cu)
    // the smallest row capacity that holds the batch (the H stages take less of the LDS)
    const bool nt = layer_bytes(n_embd, n_rows, n_vocab) > NT_BYTES;
    auto *k = n_rows <= 32    ? (nt ? k_logits32_nt : k_logits32)
              : n_rows <= 64  ? (nt ? k_logits64_nt : k_logits64)
              : n_rows <= 128 ? (nt ? k_logits128_nt : k_logits128)
                              : (nt ? k_logits256_nt : k_logits256);
    hipLaunchKernelGGL(k, dim3(grid), dim3(LNT), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        qs_set_error("output layer launch: %s", hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? QS_ENOMEM : QS_EDEVICE;
    }
    return 0;
}
