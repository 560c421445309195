// Transposing pack / unpack of views with a short side, and of small views.
//
// The tiles of transpose_kernels.hip are 256 or 512 bytes long on both sides, so a view whose memory-contiguous extent
// or whose packed rows are shorter than that (the keys of an attention layer sent as [.., head dim, sequence], a tall
// matrix of a few columns) fills only part of them, and a small view makes too few of them for 256 CUs.  Here the two
// sides of a tile have lengths of their own: 64 to 512 bytes along the short side, what a tile of 2 to 64 KiB leaves
// along the other.
//
// A tile is read as rows i of consecutive elements j and written as rows j of consecutive elements i: packing, i runs
// over q and j over the memory-contiguous dimension c; unpacking, the other way round.  HBM-bound: 2 bytes of traffic
// per byte moved.  Both sides move 16-byte vectors whatever the extents: the last vector of a row is moved back so that it
// ends where the row ends.  bf16 [64, 4096, 64] -> [64, 64, 4096] (33.6 MB), pack / unpack: 95.8 / 104 us with the tiles
// that fill a quarter of their lanes, 10.9 / 11.0 us here (6.1 TB/s); head dim 80: 98 / 82 -> 15.6 / 17.7,
// 32: 94 / 81 -> 6.5 / 6.6; u8 head dim 128: 222 / 303 -> 11.0 / 11.9; bf16 1024^2: 3.3 / 3.4 -> 2.2 / 2.2.
//
// Most launches are one or two rounds of workgroups, so what a wavefront issues before its first load and between its loads
// and its stores is not hidden: tile numbers are decoded by multiplication (FastDiv32; the compiler's 64-bit divisions were
// some 120 of 185 scalar instructions a wavefront), an address is one 32 x 32-bit multiply-add (ONE), rows and vectors of a
// pass follow from those of the pass before.  With divisions and 64-bit multiplications / now, us: f32 512^2 2.77 / 2.58,
// 1216^2 3.47 / 2.96, u8 [68359, 32, 32] 86 / 69, f32 [68359, 16, 16] 45.9 / 37, f32 [40, 2000, 128] 18.7 / 17.0, 1000 calls of all
// types and sizes 0.92 x on average.
#include <type_traits>

#include "mhip_device.h"
#include "pack_internal.h"

namespace mhip {

// What views of one dimension after c and at most one before it need (ONE), in 112 bytes: see SmallDims for why that counts.
struct NarrowOneArgs {
    char* base;                   // address of the view's first element
    char* packed;
    uint32_t Sc, Q;               // extents along c and along q
    uint32_t vi, vj;              // read rows and columns a tile holds: the tile's own, or the extent where that is shorter
    FastDiv32 nv_div;             // vectors per read row
    uint32_t row_step, vec_step;  // a pass of all lanes over the vectors of the read rows: lanes / nv and lanes % nv
    uint32_t ntiles, per_xcd;     // each XCD takes a contiguous share of the tiles
    uint32_t wg0;                 // workgroups of this copy launched before this grid
    uint32_t mem_pitch;           // consecutive q lie that many elements apart
    FastDiv32 per_batch_div;      // tiles per matrix
    FastDiv32 fast_div;           // tiles along the side that has fewer of them
    uint32_t i_fast;              // that side is i
    uint32_t write_through;       // how written vectors are stored, see try_narrow_transpose
    uint64_t batch_stride;        // bytes
};

struct NarrowArgs : NarrowOneArgs {
    int n_inner, n_outer;         // dimensions after c (q -> memory offset) and before c (batch -> memory offset)
    FastDiv32 inner_div[kMaxCanonDims];
    uint64_t inner_stride[kMaxCanonDims];  // bytes
    FastDiv32 outer_div[kMaxCanonDims];
    uint64_t outer_stride[kMaxCanonDims];  // bytes
};

// v shifted down by `bytes` < 16
__device__ __forceinline__ u32x4 shift_down(u32x4 v, uint32_t bytes) {
    if (bytes & 8u) { v.x = v.z; v.y = v.w; }
    if (bytes & 4u) { v.x = v.y; v.y = v.z; v.z = v.w; }
    const uint32_t r = bytes & 3u;
    return u32x4{__builtin_amdgcn_alignbyte(v.y, v.x, r), __builtin_amdgcn_alignbyte(v.z, v.y, r),
                 __builtin_amdgcn_alignbyte(v.w, v.z, r), v.w >> (8 * r)};
}

// TI x TJ elements.  In LDS the 16-byte groups of the read rows are numbered through, f = i * GJ + group, and permuted by
// XOR of the low four bits of f with a key of i / E.  Sixteen consecutive groups lie in one block of E read rows, so the
// key is the same for all of them and the permutation stays inside their 256 bytes, i.e. inside one turn of the banks:
//   * a lane stores its vector as one group, sixteen lanes a whole turn, whatever the key;
//   * on the way out a lane collects E elements of one column from E consecutive read rows, as 32-bit words (narrower
//     elements: 2 or 4 columns at once, sorted out in registers).  The NIV lanes that take different blocks of one column
//     see different keys (M apart), the 64 / NIV word columns beside them fill the rest of the turn: while the read rows
//     are whole blocks, no two of the 64 lanes meet in a bank at different addresses.  The last vector of a ragged row
//     starts inside a block and sees two keys, i.e. up to two addresses in a bank; words of 8 bytes take two turns anyway,
//     three when ragged.
// As many wavefronts per SIMD as the tiles that fit the 160 KiB of LDS bring, eight at most: the registers must not allow fewer.
// (Left alone, the compiler moves the LDS reads of all passes of a 64 KiB tile ahead, in 230 registers: one workgroup per CU
// and 19 us where two take 11.)  Where LATE it is left alone: all columns are collected before the first is stored (see
// launch_narrow_tile).
constexpr int narrow_waves(int threads, int tile_bytes, bool late) {
    const int waves = 163840 / tile_bytes * threads / 256;
    return late ? 1 : waves > 8 ? 8 : waves;
}

template <typename T, int THREADS, bool PACK, int TI, int TJ, bool ONE, bool LATE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(narrow_waves(THREADS, TI * TJ * sizeof(T), LATE), 8)))
void slice_transpose_narrow_kernel(std::conditional_t<ONE, NarrowOneArgs, NarrowArgs> a) {
    constexpr uint32_t ES = sizeof(T), E = 16 / ES;
    constexpr uint32_t GJ = TJ / E, GI = TI / E;
    constexpr uint32_t W = ES >= 4 ? 1 : 4 / ES;  // columns per LDS word
    constexpr uint32_t NIV = GI >= 16 ? 16 : GI, M = 16 / NIV;
    static_assert(TI % E == 0 && TJ % E == 0 && TJ >= 16 && (TI * GJ) % 16 == 0, "whole turns of the permutation");
    constexpr uint32_t RP = TI * GJ / THREADS;             // load passes
    constexpr uint32_t WP = GI * (TJ / W) / THREADS;       // store passes
    static_assert(RP * THREADS == TI * GJ && WP * THREADS == GI * (TJ / W) && GI % NIV == 0, "whole passes");
    using Word = typename UnitType<(ES >= 4 ? ES : 4)>::type;
    __shared__ __attribute__((aligned(16))) char tile[TI * TJ * ES];

    const uint32_t wg = a.wg0 + blockIdx.x;
    const uint32_t id = (wg & 7) * a.per_xcd + (wg >> 3);
    if (id >= a.ntiles) return;
    uint32_t b, in_batch, slow, fast;
    a.per_batch_div.divmod(id, b, in_batch);
    // the side with fewer tiles is the fast one: neighbouring workgroups share whole rows of it
    a.fast_div.divmod(in_batch, slow, fast);
    // a tile that would hang over the edge is moved back inside; the overlap is written twice, same bytes
    const uint32_t I = PACK ? a.Q : a.Sc, J = PACK ? a.Sc : a.Q;
    uint32_t i0 = (a.i_fast ? fast : slow) * TI, j0 = (a.i_fast ? slow : fast) * TJ;
    if (i0 + a.vi > I) i0 = I - a.vi;
    if (j0 + a.vj > J) j0 = J - a.vj;
    const uint32_t q0 = PACK ? i0 : j0, c0 = PACK ? j0 : i0;
    char* __restrict__ packed = a.packed + (((uint64_t)b * a.Sc + c0) * a.Q + q0) * ES;  // the tile's first element, on both sides
    char* __restrict__ mem = a.base + (uint64_t)c0 * ES;
    if constexpr (ONE) {
        mem += b * a.batch_stride + (uint64_t)q0 * a.mem_pitch * ES;
    } else {
        for (int k = a.n_outer - 1; k >= 0; --k) {
            uint32_t rest, index;
            a.outer_div[k].divmod(b, rest, index);
            mem += index * a.outer_stride[k];
            b = rest;
        }
    }
    // addresses inside the tile: q and c counted from its first element
    auto packed_at = [&](uint32_t q, uint32_t c) { return packed + ((uint64_t)c * a.Q + q) * ES; };
    auto mem_at = [&](uint32_t q, uint32_t c) {
        if constexpr (ONE) {
            return mem + ((uint64_t)q * a.mem_pitch + c) * ES;
        } else {
            uint64_t off = 0;
            uint32_t rest = q0 + q;
            for (int k = a.n_inner - 1; k > 0; --k) {
                uint32_t qd, r;
                a.inner_div[k].divmod(rest, qd, r);
                off += (uint64_t)r * a.inner_stride[k];
                rest = qd;
            }
            return mem + (off + (uint64_t)rest * a.inner_stride[0] + (uint64_t)c * ES);
        }
    };

    // ---- read side -> LDS: the tile's vectors numbered through, so that short rows leave no lane idle ----
    const uint32_t nv = a.nv_div.d, total = a.vi * nv;
    const bool ragged_j = a.vj % E != 0;
    u32x4 d[RP];
    uint32_t row[RP], vec[RP];
    a.nv_div.divmod(threadIdx.x, row[0], vec[0]);
#pragma unroll
    for (uint32_t p = 0; p < RP; ++p) {
        if (p > 0) {  // every pass moves on by the same number of vectors
            row[p] = row[p - 1] + a.row_step;
            vec[p] = vec[p - 1] + a.vec_step;
            if (vec[p] >= nv) {
                vec[p] -= nv;
                ++row[p];
            }
        }
        if (p * THREADS < total) {
            const uint32_t r = row[p] < a.vi ? row[p] : a.vi - 1;  // no load is predicated
            uint32_t col = vec[p] * E;
            if (ragged_j) col = col + E <= a.vj ? col : a.vj - E;
            const uint4 v = load16_unaligned(PACK ? mem_at(r, col) : packed_at(col, r));
            d[p] = u32x4{v.x, v.y, v.z, v.w};
        }
    }
#pragma unroll
    for (uint32_t p = 0; p < RP; ++p) {
        const uint32_t r = row[p], g = vec[p];
        if (r < a.vi) {
            u32x4 v = d[p];
            if (ragged_j) v = shift_down(v, g * E + E <= a.vj ? 0u : (g * E + E - a.vj) * ES);  // a vector that was moved back
            const uint32_t f = (r * GJ + g) ^ (((r / E) * M) & 15u);
            *reinterpret_cast<u32x4*>(tile + f * 16) = v;
        }
    }
    __syncthreads();

    // ---- LDS -> written side ----
    const bool ragged_i = a.vi % E != 0;
#pragma unroll
    for (uint32_t p = 0; p < WP; ++p) {
        const uint32_t u = threadIdx.x + p * THREADS;
        const uint32_t rest = u / 64;
        const uint32_t iv = u % NIV + NIV * (rest % (GI / NIV));                               // block of E read rows
        const uint32_t j = ((rest / (GI / NIV)) * (64 / NIV) + (u % 64) / NIV) * W;            // first column of the word
        if (j < a.vj && iv * E < a.vi) {
            const uint32_t g = j / E, byte = (j % E) * ES;
            Word w[E];
            uint32_t i = iv * E;
            if (!ragged_i) {
                // within a block the rows' groups differ from the first row's by XOR with a constant
                const uint32_t first = (((E * iv * GJ + g) ^ ((iv * M) & 15u)) * 16) + byte;
#pragma unroll
                for (uint32_t k = 0; k < E; ++k)
                    w[k] = *reinterpret_cast<const Word*>(tile + (GJ >= 16 ? first + k * GJ * 16 : first ^ (k * GJ * 16)));
            } else {
                if (i + E > a.vi) i = a.vi - E;  // the last vector of a written row, moved back
#pragma unroll
                for (uint32_t k = 0; k < E; ++k) {
                    const uint32_t r = i + k;
                    w[k] = *reinterpret_cast<const Word*>(tile + ((r * GJ + g) ^ (((r / E) * M) & 15u)) * 16 + byte);
                }
            }
            u32x4 out[W];
            if constexpr (ES == 8) {
                out[0] = u32x4{(uint32_t)w[0], (uint32_t)(w[0] >> 32), (uint32_t)w[1], (uint32_t)(w[1] >> 32)};
            } else if constexpr (ES == 4) {
                out[0] = u32x4{w[0], w[1], w[2], w[3]};
            } else if constexpr (ES == 2) {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    out[0][k] = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x05040100u);
                    out[1][k] = __builtin_amdgcn_perm(w[2 * k + 1], w[2 * k], 0x07060302u);
                }
            } else {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {  // four rows of four bytes, transposed
                    const uint32_t ab_lo = __builtin_amdgcn_perm(w[4 * k + 1], w[4 * k], 0x05010400u);
                    const uint32_t ab_hi = __builtin_amdgcn_perm(w[4 * k + 1], w[4 * k], 0x07030602u);
                    const uint32_t cd_lo = __builtin_amdgcn_perm(w[4 * k + 3], w[4 * k + 2], 0x05010400u);
                    const uint32_t cd_hi = __builtin_amdgcn_perm(w[4 * k + 3], w[4 * k + 2], 0x07030602u);
                    out[0][k] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);
                    out[1][k] = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);
                    out[2][k] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
                    out[3][k] = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < W; ++k) {
                if (k == 0 || j + k < a.vj) {
                    char* dst = PACK ? packed_at(i, j + k) : mem_at(j + k, i);
                    if (a.write_through) store16_writethrough_raw(dst, out[k]);  // wave-uniform
                    else *reinterpret_cast<u32x4_unaligned*>(dst) = out[k];
                }
            }
        }
    }
}

// Returned instead of a status for a view of too many tiles: the caller leaves the view to another kernel.
constexpr int kTooManyTiles = -1;

// WB and RB: bytes of a written and of a read row of the tile; GENERAL: addresses by the general form for every view (see
// launch_narrow_tile)
template <typename T, bool PACK, int WB, int RB, bool LATE = false, bool GENERAL = false>
static int launch_narrow(NarrowArgs& a, uint64_t nbatch, hipStream_t stream) {
    constexpr uint32_t ES = sizeof(T), E = 16 / ES, TI = WB / ES, TJ = RB / ES;
    constexpr int kBytes = TI * TJ * ES, kLanes = kBytes >= 32768 ? 512 : kBytes >= 8192 ? 256 : 128;
    const uint32_t I = PACK ? a.Q : a.Sc, J = PACK ? a.Sc : a.Q;
    a.vi = I < TI ? I : TI;
    a.vj = J < TJ ? J : TJ;
    const uint32_t ti_count = (I + TI - 1) / TI, tj_count = (J + TJ - 1) / TJ, nv = (a.vj + E - 1) / E;
    a.nv_div = FastDiv32(nv);
    a.row_step = kLanes / nv;
    a.vec_step = kLanes % nv;
    // The kernel's tile numbers, up to 7 past the last one, are dividends of FastDiv32.  A tile holds 128 bytes at least (8 x 8
    // elements of 2 bytes), so a view of 256 GiB can have more of them.
    const uint64_t ntiles = nbatch * ti_count * tj_count;
    if (ntiles >= kFastDivLimit - 8) return kTooManyTiles;
    a.ntiles = (uint32_t)ntiles;
    a.per_xcd = (a.ntiles + 7) / 8;
    a.per_batch_div = FastDiv32(ti_count * tj_count);
    a.i_fast = ti_count < tj_count;
    a.fast_div = FastDiv32(a.i_fast ? ti_count : tj_count);
    const bool one = a.n_inner == 1 && a.n_outer <= 1 && a.inner_stride[0] / ES <= UINT32_MAX;
    a.mem_pitch = (uint32_t)(a.inner_stride[0] / ES);
    a.batch_stride = a.n_outer == 1 ? a.outer_stride[0] : 0;
    return launch_in_pieces((uint64_t)a.per_xcd * 8, kLanes, 8, [&](uint64_t wg0, uint32_t count) {
        a.wg0 = (uint32_t)wg0;
        if constexpr (!GENERAL) {
            if (one) {
                const NarrowOneArgs& small = a;
                MHIP_LAUNCH((slice_transpose_narrow_kernel<T, kLanes, PACK, TI, TJ, true, LATE>), dim3(count), dim3(kLanes), 0, stream, small);
                return;
            }
        }
        MHIP_LAUNCH((slice_transpose_narrow_kernel<T, kLanes, PACK, TI, TJ, false, LATE>), dim3(count), dim3(kLanes), 0, stream, a);
    });
}

// The same with tiles that are longer along the long side (the written rows where LONG_I, else the read rows), where that
// pays.  It does in two cases:
//   * 400 to 512 tiles of 64 KiB (two fit a CU's LDS; the numbers stand for the 256 CUs of the whole part, on fewer the choice only
//     costs time): all of them are resident at once, so the part first reads everything and then writes everything, in pieces of
//     1 KiB and more, and no write gets between the reads.  2- and 4-byte elements, packing / unpacking, small tiles -> 64 KiB, us:
//     bf16 [64, 4096, 64] 13.4 / 12.9 -> 10.9 / 11.0, [56, 4096, 64] 12.4 / 13.1 -> 10.1 / 10.1, [256, 1024, 64] 13.9 / 12.7 -> 11.0 /
//     11.6, f32 [262144, 32] 14.1 / 12.5 -> 11.2 / 10.9.  With more of them the part runs out of step again and large tiles lose
//     ([96, 4001, 64] 19.2 / 18.0 -> 20.8 / 20.0); with half as many they are within 4 % either way ([32, 4096, 64] 6.5 / 6.5 -> 6.3 / 6.4;
//     the first line was measured at 8.1 / 7.5 and 8.8 / 8.4, with addresses in 64 bits).
//   * 4-byte elements from 28 MiB on: tiles of 32 KiB instead of 16 ([1 M, 16] 28.0 / 25.8 -> 24.7 / 23.2 and others 0.89 to 0.99 x
//     with addresses in 64 bits, 17 MiB up to 1.1 x; with the present ones 24.6 / 23.6 -> 24.8 / 23.1, nothing more than 4 % either way).
constexpr uint64_t kResidentTilesMin = 400, kResidentTilesMax = 512;
template <typename T, bool PACK, int WB, int RB, bool LONG_I>
static int launch_narrow_long(NarrowArgs& a, uint64_t nbatch, hipStream_t stream) {
    constexpr int ES = sizeof(T), K = 65536 / (WB * RB / ES);  // times as long: a tile of 64 KiB
    const uint32_t I = PACK ? a.Q : a.Sc, J = PACK ? a.Sc : a.Q;
    // whether the long side fills most of a tile that is `k` times as long
    auto fills = [&](int k) { return (uint64_t)(LONG_I ? I : J) * ES * 4 >= (uint64_t)(LONG_I ? WB : RB) * k * 3; };
    if constexpr (ES == 2 || ES == 4) {
        constexpr uint32_t TI = WB / ES * (LONG_I ? K : 1), TJ = RB / ES * (LONG_I ? 1 : K);
        const uint64_t tiles = nbatch * ((I + TI - 1) / TI) * ((J + TJ - 1) / TJ);
        if (fills(K) && tiles >= kResidentTilesMin && tiles <= kResidentTilesMax)
            return launch_narrow<T, PACK, WB * (LONG_I ? K : 1), RB * (LONG_I ? 1 : K)>(a, nbatch, stream);
    }
    if constexpr (ES == 4)
        if (fills(2) && nbatch * I * J * ES >= (28ull << 20))
            return launch_narrow<T, PACK, WB * (LONG_I ? 2 : 1), RB * (LONG_I ? 1 : 2)>(a, nbatch, stream);
    return launch_narrow<T, PACK, WB, RB>(a, nbatch, stream);
}

// Tile length along a side of `bytes` <= 512: pieces of 128 bytes where they cover the side with little overlap (the last
// one is moved back), else the next power of two (272 bytes, 67 MB, pack / unpack: one tile of 512 26 / 27 us, three
// of 128 47 / 29; 384 bytes: 27.8 / 25 against 27.5 / 24.5).
static uint32_t narrow_tile_bytes(uint64_t bytes) {
    if (bytes <= 64) return 64;
    if (bytes <= 128) return 128;
    const uint64_t pieces = (bytes + 127) / 128 * 128;
    return pieces * 10 <= bytes * 11 ? 128 : bytes <= 256 ? 256 : 512;
}

// Which tile: from 16 MiB on, the short side's length from narrow_tile_bytes and the other side's so that the two lengths
// multiply to 64 KiB (tiles of 64, 32, 16, 8 KiB of 1-, 2-, 4-, 8-byte elements); below that 128 x 128 bytes, which makes
// more workgroups (bf16 16384 x 20: 2.4 us against 3.0, 65536 x 64 (8.4 MB) 3.6 against 3.8; 16.8 MB of keys of 64 bytes
// 8.6 against 7.5, of u8 keys of 64 bytes 8.6 against 7.5).  Of 8-byte elements that tile is 16 x 16 in 2 KiB: matrices of
// 4 MiB and more whose sides are both longer than 512 bytes take 256 x 256 bytes (f64 pack / unpack, 128 x 128 and 256 x 256: 627^2
// 3.1 / 3.3 and 2.9 / 2.9, 640^2 3.1 / 3.2 and 3.3 / 3.1, 887^2 4.8 / 5.1 and 4.0 / 3.9, 1145^2 6.7 / 6.5 and 5.8 / 5.7, where the
// tiles of transpose_kernels.hip take 6.0 / 6.0; [3584, 16, 16] 4.5 / 4.4 and 6.5 / 6.4).
// Byte matrices of more than 768 tiles (three on each of 256 CUs) and up to 23 MiB collect all columns of a tile before they store the
// first (LATE) and keep the general form of addresses (GENERAL), whose arithmetic spaces the stores: in the short form they leave
// in bursts, which pays while all tiles are in flight together and makes some shapes pay beyond.  Against 64-bit tile numbers,
// random shapes, warm and cold: up to 768 tiles the short form takes 0.85 and 0.84 of the time, 0.93 at most (LATE and GENERAL 0.96,
// 1.04 at most); 769 to 1000 tiles 0.985, but 1.05 to 1.20 on single shapes ([2049, 6001] unpack 8.6 -> 9.9 us), with LATE and
// GENERAL 0.955, 0.976 at most; 20 to 23 MiB LATE alone 0.98 and 0.99, 1.05 at most, both 0.96, 1.02 at most.  Above 23 MiB, tiles of
// 256 x 256 and GENERAL alone: 0.976 and 0.968, 1.04 at most, where the short form takes 0.977 with single shapes at 1.14 and 1.09
// ([1672, 15051] unpack 11.8 -> 13.4 us, general 12.1).
// Batches of matrices that fit 128 x 128 bytes keep that tile at any size: u8 [78125, 16, 16] 94 / 95 us, in tiles of 1024 x 64 of
// which one matrix fills little 335 / 333; bf16 [39062, 16, 16] 45 / 46 and 97 / 98, [8544, 64, 64] 23.2 / 23.3 and 30.2 / 31.3.
template <typename T, bool PACK>
static int launch_narrow_tile(NarrowArgs& a, uint64_t nbatch, hipStream_t stream) {
    constexpr uint32_t ES = sizeof(T);
    const uint64_t ib = (uint64_t)(PACK ? a.Q : a.Sc) * ES, jb = (uint64_t)(PACK ? a.Sc : a.Q) * ES;
    const uint64_t bytes = nbatch * ib * jb / ES;
    if constexpr (ES == 1)
        if (ib > 512 && jb > 512) {
            if (bytes > (23ull << 20)) return launch_narrow<T, PACK, 256, 256, false, true>(a, nbatch, stream);
            if (nbatch * ((ib + 127) / 128) * ((jb + 127) / 128) > 768) return launch_narrow<T, PACK, 128, 128, true, true>(a, nbatch, stream);
        }
    if (bytes >= (16ull << 20) && (ib <= 512 || jb <= 512) && (ib > 128 || jb > 128)) {  // a long side to fill the tile with
        const bool short_j = jb <= ib;
        uint32_t n = narrow_tile_bytes(short_j ? jb : ib);
        if (ES == 8 && n == 64) n = 128;  // a read row of 64 bytes would be fewer than 16 elements
        if (short_j) {
            if constexpr (ES < 8)
                if (n == 64) return launch_narrow_long<T, PACK, 1024, 64, true>(a, nbatch, stream);
            if (n == 128) return launch_narrow_long<T, PACK, 512, 128, true>(a, nbatch, stream);
            if (n == 256) return launch_narrow_long<T, PACK, 256, 256, true>(a, nbatch, stream);
            return launch_narrow<T, PACK, 128, 512>(a, nbatch, stream);
        }
        if constexpr (ES < 8)
            if (n == 64) return launch_narrow_long<T, PACK, 64, 1024, false>(a, nbatch, stream);
        if (n == 128) return launch_narrow_long<T, PACK, 128, 512, false>(a, nbatch, stream);
        if (n == 256) return launch_narrow_long<T, PACK, 256, 256, false>(a, nbatch, stream);
        return launch_narrow<T, PACK, 512, 128>(a, nbatch, stream);
    }
    if constexpr (ES == 8)
        if (bytes >= (4ull << 20) && ib > 512 && jb > 512) return launch_narrow<T, PACK, 256, 256>(a, nbatch, stream);
    return launch_narrow<T, PACK, 128, 128>(a, nbatch, stream);
}

// Takes the view when one of its sides is at most 512 bytes long (bf16 67 MB, sides of 512 / 768 bytes, pack: 23.8 / 27 us
// here against 24.0 / 25.4 with the long tiles; rows that are not whole lines 26.6 against 34.3, and 27 against 25.4) or
// when it has at most 12 MiB (bf16 2048^2 3.6 us against 4.0, 2000 x 3000 6.9 against 8.4, u8 2000 x 3000 4.4 against
// 6.2; fp32 2000 x 3000, 24 MB, 11 against 10.4), both sides holding at least one vector.  Byte matrices whose rows are not
// whole cache lines are taken up to 40 MiB, in tiles of 128 x 128 up to 23 MiB and of 256 x 256 above: the strips of the other
// file need more of them to fill the part, its fixed tiles share lines.  Fixed tiles / 128 x 128 / 256 x 256, packing, over
// 700 MB of buffers: 4097^2 16.2 / 11.8 / 15.2 us, 4803^2 17.5 / 13.6 / 16.2, 5017^2 18.2 / 15.9 / 16.3, 5616^2 21.3 / 17.3 / 15.3,
// 6395^2 28.7 / 26.1 / 24.0 (7000^2, 47 MiB, 30.3 with the fixed tiles and 31.5 with 256 x 256; 4096^2, whole lines, 7.2 and 7.7).
// Over three sets of buffers, which the Infinity Cache holds: 11.3 / 10.4 / 13.6, 12.1 / 13.0 / 15.1, 12.4 / 15.7 / 15.9, 18.0 / 17.1 /
// 13.7, 20.7 / 25.4 / 23.0, so above 23 MiB copies between cached buffers lose up to a third and the others gain as much.
template <bool PACK>
bool try_narrow_transpose(char* base, char* packed, const CanonSlice& c, int cd, uint64_t nbatch, uint32_t Q, uint32_t unit,
                          hipStream_t stream, int* rc) {
    const uint64_t Sc = c.dims[cd].size, bytes = nbatch * Sc * Q * unit;
    const uint64_t short_side = (Sc < Q ? Sc : Q) * unit;
    if (unit > 8 || short_side < 16) return false;
    if (short_side > 512 && bytes > (unit == 1 ? 40ull << 20 : 12ull << 20)) return false;
    NarrowArgs a{};
    uint64_t written = PACK ? (uint64_t)(uintptr_t)packed | (uint64_t)Q * unit : (uint64_t)(uintptr_t)(base + c.offset * unit);
    for (int k = 0; k < c.ndim; ++k) {
        if (k == cd) continue;
        const uint64_t stride = c.dims[k].stride * unit;
        if (k > cd) {
            a.inner_div[a.n_inner] = FastDiv32((uint32_t)c.dims[k].size);
            a.inner_stride[a.n_inner++] = stride;
        } else {
            a.outer_div[a.n_outer] = FastDiv32((uint32_t)c.dims[k].size);
            a.outer_stride[a.n_outer++] = stride;
        }
        if (!PACK) written |= stride;
    }
    if (short_side > 512 && bytes > (12ull << 20)) {  // bytes, see above
        uint64_t rows = (uint64_t)(uintptr_t)packed | Q | (uint64_t)(uintptr_t)(base + c.offset);
        for (int k = 0; k < c.ndim; ++k)
            if (k != cd) rows |= c.dims[k].stride;
        if ((rows & 127u) == 0) return false;
    }
    a.base = base + c.offset * unit;
    a.packed = packed;
    a.Sc = (uint32_t)Sc;
    a.Q = Q;
    // Written rows that start on half cache lines are stored write-through (33.6 MB of keys 10.9 us against 12.3 through the
    // cache, unpacked rows of 64 bytes 6.6 against 7.7); others go through the cache, which combines what neighbouring
    // tiles share (rows of 4001 bf16 19.1 against 21.0, unpacked rows of 160 bytes 17.7 against 18.4), unless the launch
    // is small enough to be bound by latency (bf16 1500^2 3.1 against 3.2).
    a.write_through = (written & 63u) == 0 || bytes <= (8ull << 20);
    switch (unit) {
        case 1: *rc = launch_narrow_tile<uint8_t, PACK>(a, nbatch, stream); break;
        case 2: *rc = launch_narrow_tile<uint16_t, PACK>(a, nbatch, stream); break;
        case 4: *rc = launch_narrow_tile<uint32_t, PACK>(a, nbatch, stream); break;
        default: *rc = launch_narrow_tile<uint64_t, PACK>(a, nbatch, stream); break;
    }
    return *rc != kTooManyTiles;
}

template bool try_narrow_transpose<true>(char*, char*, const CanonSlice&, int, uint64_t, uint32_t, uint32_t, hipStream_t, int*);
template bool try_narrow_transpose<false>(char*, char*, const CanonSlice&, int, uint64_t, uint32_t, uint32_t, hipStream_t, int*);

}  // namespace mhip
