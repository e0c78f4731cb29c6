// qs_logits.hip - the output layer alone: logits[r][v] = sum_k H[r][k] W[v][k], bf16 operands
// and fp32 accumulation on the matrix cores (forward_cpu.c:319-323 at bf16), for up to 256
// rows against the weights packed by k_head_pack.
//
// What bounds it: W (2 V E bytes) is read from HBM once and the logits (4 V rows) are written
// once; at 256 rows x 2048 x 151,936 that is 622 + 156 MB against 159 GFLOP, so the layer
// streams.  W reaches the CUs at (bytes in flight) / (load latency), and every CU has to
// stream until the end.  Hence:
//
//   * One workgroup of 8 wavefronts per CU, all of a CU's 160 KB of LDS: a ring of H stages
//     (from the XCD's L2, short latency) three deep and a ring of W stages (HBM) seven to
//     nine deep.  Loads return in order per wavefront, so the two rings belong to different
//     wavefronts: 0-3 load H, 4-7 load W, each waits for its own, and the stage's barrier
//     joins them.  Six or more W stages of 16 KB stay in flight a CU; the earlier shape (two
//     workgroups a CU, three shared stages) held 32 KB.
//   * The vocabulary is dealt out in 32-column blocks, an equal run for each workgroup (18 or
//     19 blocks at V = 151,936 on 256 CUs).  One 128-column tile per workgroup made 1,187
//     workgroups for 512 places: a third round with two thirds of the chip idle.
//   * A run is cut into tiles of at most 8 blocks whose stages follow each other in the rings
//     without a break: while a tile's accumulators are stored, the next tile's loads are in
//     flight.  The stores go straight from the accumulators (32 lanes, 128 consecutive bytes
//     a row), with no LDS and no barrier.
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
template <> struct LinShape<128> { static constexpr int WRB = 2, RG = 2, CG = 4, TB = 10, HS = 3, WS = 6; };
template <> struct LinShape<64> { static constexpr int WRB = 2, RG = 1, CG = 8, TB = 10, HS = 3, WS = 7; };
template <> struct LinShape<32> { static constexpr int WRB = 1, RG = 1, CG = 8, TB = 10, HS = 3, WS = 7; };

// 64 bytes a row or column, its four 16-byte segments stored in the order
// seg ^ ((row / 4) % 4): the lanes of an operand read hit distinct banks.
template <int RB>
struct LinLds {
    uint16_t h[LinShape<RB>::HS][RB][LK];
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

// The same for a count known at run time: N stages of c loads each, 1 <= c <= 5 (uniform).
template <int N>
__device__ __forceinline__ void vm_wait_stages(int c) {
    switch (c) {
    case 1: vm_wait<N>(); break;
    case 2: vm_wait<2 * N>(); break;
    case 3: vm_wait<3 * N>(); break;
    case 4: vm_wait<4 * N>(); break;
    default: vm_wait<5 * N>(); break;
    }
}

template <int RB>
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
    const int total = ntile * nst;                  // stages of the run
    // tile t of the run: blocks [tile_begin(t), tile_begin(t + 1))
    const int per = nbk / ntile, extra = nbk - per * ntile;
    auto tile_begin = [&](int t) { return b0 + per * t + min(t, extra); };
    const int wc = (per + 1) / 2;                   // W pieces of a wavefront per stage, at
                                                    // least (its tiles hold per or per + 1)

    const bool wload = wv >= 4;                     // this wavefront loads W (else H)
    const bool hload = !wload && wv < HPIECES;
    // the load side: the next stage's tile and stage within it, its ring slot, and where the
    // wavefront's pieces of the tile start (one per lane: H; uniform: W)
    int lt = 0, ls = 0, lslot = 0;
    uint32_t hoff[HL];                              // bytes
    uint32_t woff[WL];                              // KB (a packed piece is 1 KB)
#pragma unroll
    for (int i = 0; i < HL; ++i) {                  // rows 16 p .. + 16; rows past the batch
        const int r = (wv + 4 * i) * 16 + (lane >> 2);   // read row 0 (never used)
        hoff[i] = 2u * (uint32_t)((r < B ? r : 0) * E + ((lane & 3) ^ ((r >> 2) & 3)) * 8);
    }
    int lc = 0;                                     // W pieces it loads per stage of the tile
    auto load_tile = [&]() {
        // piece p: 16 columns (1 KB, packed contiguously and already swizzled); the last
        // wavefronts' surplus pieces of an odd share read piece 0 again (cached)
        const int tb = tile_begin(lt), nb = tile_begin(lt + 1) - tb;
        lc = (nb + 1) / 2;
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int p = (wv & 3) + 4 * i;
            const int col = tb * 32 + (p < 2 * nb ? p * 16 : 0);
            woff[i] = (uint32_t)__builtin_amdgcn_readfirstlane(col / LT * nst * 8 + col % LT / 16);
        }
    };
    load_tile();
    auto issue = [&]() {
        if (wload) {
#pragma unroll
            for (int i = 0; i < WL; ++i) {
                if (i >= lc) break;                 // (uniform)
                __builtin_amdgcn_global_load_lds(
                    (const char *)a.w + ((uint64_t)(woff[i] + (uint32_t)ls * 8u) << 10) +
                        (uint32_t)(lane * 16),
                    &L.w[lslot][((wv & 3) + 4 * i) * 16][0], 16, 0, 2);
            }
            lslot = lslot + 1 == WS ? 0 : lslot + 1;
        } else if (hload) {
#pragma unroll
            for (int i = 0; i < HL; ++i)
                __builtin_amdgcn_global_load_lds((const char *)(a.h + ls * LK) + hoff[i],
                                                 &L.h[lslot][(wv + 4 * i) * 16][0], 16, 0, 0);
            lslot = lslot + 1 == HS ? 0 : lslot + 1;
        }
        if (++ls == nst) {
            ls = 0;
            ++lt;
            load_tile();
        }
    };
    const int depth = wload ? WS - 1 : HS - 1;      // stages in flight ahead of the products
    for (int g = 0; g < depth && g < total; ++g) issue();

    // wavefront w: rows 32 WRB (w % RG) .. + 32 WRB; blocks w / RG + CG j of a tile
    const int rg = wv % RG, cg = wv / RG;
    const int rr = lane & 31, swz = (rr >> 2) & 3;
    int g = 0, hslot = 0, wslot = 0;
    auto tile = [&](auto nbc, int tb) __attribute__((always_inline)) {
        constexpr int NBW = decltype(nbc)::value;   // this wavefront's blocks
        f32x16 acc[WRB][NBW > 0 ? NBW : 1];
#pragma unroll
        for (int i = 0; i < WRB; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j) acc[i][j] = f32x16{};
        for (int st = 0; st < nst; ++st, ++g) {
            // this stage's own loads are in (the later stages' stay in flight; stores of an
            // earlier tile among them only make the wait longer)
            if (g + depth < total + 1) {
                if (wload) vm_wait_stages<WS - 2>(wc);
                else vm_wait<(HS - 2) * HL>();
            } else {
                vm_wait<0>();
            }
            // the slots refilled next were read before this barrier by every wavefront
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (g + depth < total) issue();
            const uint16_t(*hs)[LK] = L.h[hslot];
            const uint16_t(*ws)[LK] = L.w[wslot];
            hslot = hslot + 1 == HS ? 0 : hslot + 1;
            wslot = wslot + 1 == WS ? 0 : wslot + 1;
            if constexpr (NBW > 0) {
#pragma unroll
                for (int ks = 0; ks < LK / 16; ++ks) {
                    const int sg = ((ks * 2 + (lane >> 5)) ^ swz) * 8;
                    u32x4 ha[WRB], wb[NBW];
#pragma unroll
                    for (int i = 0; i < WRB; ++i)
                        ha[i] = *(const u32x4 *)&hs[(rg * WRB + i) * 32 + rr][sg];
#pragma unroll
                    for (int j = 0; j < NBW; ++j)
                        wb[j] = *(const u32x4 *)&ws[(cg + CG * j) * 32 + rr][sg];
#pragma unroll
                    for (int j = 0; j < NBW; ++j)
#pragma unroll
                        for (int i = 0; i < WRB; ++i)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                __builtin_bit_cast(bf16x8, ha[i]),
                                __builtin_bit_cast(bf16x8, wb[j]), acc[i][j], 0, 0, 0);
                }
            }
        }
        // lane l, element q of an accumulator: row (q / 4) * 8 + (l / 32) * 4 + q % 4 of the
        // block, column l % 32
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const int col = (tb + cg + CG * j) * 32 + rr;
#pragma unroll
            for (int i = 0; i < WRB; ++i) {
                const int r0 = (rg * WRB + i) * 32 + (lane >> 5) * 4;
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int r = r0 + (q >> 2) * 8 + (q & 3);
                    if (r < B && col < V) a.logits[(int64_t)r * V + col] = acc[i][j][q];
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
}

// One kernel per shape (a template kernel's host stub is not emitted here).
__global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_logits32(LinArgs a) { lin_run<32>(a); }
__global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_logits64(LinArgs a) { lin_run<64>(a); }
__global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_logits128(LinArgs a) { lin_run<128>(a); }
__global__ void __launch_bounds__(LNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_logits256(LinArgs a) { lin_run<256>(a); }

}  // namespace

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
    const unsigned grid = (unsigned)(a.nblk < n_cu ? a.nblk : n_cu);
    // the smallest row capacity that holds the batch (the H stages take less of the LDS)
    hipLaunchKernelGGL(n_rows <= 32    ? k_logits32
                       : n_rows <= 64  ? k_logits64
                       : n_rows <= 128 ? k_logits128
                                       : k_logits256,
                       dim3(grid), dim3(LNT), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        qs_set_error("output layer launch: %s", hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? QS_ENOMEM : QS_EDEVICE;
    }
    return 0;
}
