/**
 *  @brief gfx950 (MI355X, CDNA4) kernels for packed batched dot products: C = A * B^T.
 *  @file numkong_amd/csrc/dots_gfx950.hpp
 *
 *  Everything the HIP translation units share: the packed image, the packing kernels, the element types and the
 *  product kernel with its launch logic. dots_gfx950.hip holds the plain-C entry points of <numkong_amd/hip_abi.h>;
 *  dots_gfx950_<T>.hip instantiate the product kernels of one element type each, so that they compile side by side.
 *
 *  Replaces the per-ISA kernels the reference instantiates from
 *  include/numkong/dots/serial.h:245-333 (pack size, pack) and :520-1072 (packed product) for
 *  i8, u8, bf16, f16, e4m3, e5m2.
 *
 *  Packed image of B (n rows of k elements), all little-endian:
 *
 *      [ 64-byte header ][ tiles ][ per-column compensation terms, u32 x 32 x n_tiles ]
 *
 *  A "chunk" is 16 consecutive bytes of one B row (16 i8/fp8 values, 8 bf16/f16 values). Rows are grouped
 *  into tiles of 32; K is padded with zeros to a multiple of 8 chunks (128 bytes) and N with zero rows to
 *  a multiple of 32. Chunk `c` of row `r` of tile `t` lives at
 *
 *      data + ((t * k_chunks + c) * 32 + r) * 16
 *
 *  so the 64 lanes of a wavefront that execute one 32x32 MFMA step `q` (lane l supplies row l % 32 and
 *  chunk 2q + l / 32) read 1024 contiguous bytes at `data + (t * k_chunks + 2q) * 512 + l * 16`: the image
 *  is the MFMA operand-fragment order, and B goes from HBM to registers with one coalesced 128-bit load
 *  per lane per step, never through LDS. Which k sits in which operand slot of the instruction does not
 *  matter as long as A and B agree, and they do: A fragments are read from LDS with the same rule.
 *  e4m3, e5m2 and e3m2 are stored widened to f16 (see packed_bytes_of), so their chunks hold 8 values.
 *
 *  u8 has no unsigned MFMA. B is stored as b' = b ^ 0x80 (signed b - 128), A is turned into
 *  a' = a ^ 0x80 on its way into LDS, and  sum(a*b) = sum(a'*b') + 128*sum(a) + 128*sum(b')  (mod 2^32)
 *  with zero padding contributing nothing. 128*sum(b') per column is stored behind the tiles at pack
 *  time; sum(a) per row is accumulated with v_sad_u8 while A is staged.
 */#ifndef NUMKONG_AMD_DOTS_GFX950_HPP
#define NUMKONG_AMD_DOTS_GFX950_HPP

#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "numkong_amd/hip_abi.h"

/** What crosses translation units: the product's arguments, its scratch memory, one launcher per element type. */
namespace nk_gfx950 {

// Tile rows per band of the walk over the tile grid. An XCD works on 32 tiles at a time, a band's height times as many
// columns: 8 x 4 is the shape with the smallest perimeter for the 256 x 256 and the 128 x 256 tile alike, and the
// perimeter is what the XCD's L2 fetches per sweep of the depth (measured at 8192^3, bytes read per launch: bf16 2.18 GB
// with 8, 2.75 GB with 4 or 16, 5.28 GB with 2; i8 0.82 GB with 8 or 4, 1.22 GB with 2 or 16). NK_TILE_BAND overrides it
// for such measurements (make EXTRA=-DNK_TILE_BAND=4).
#ifndef NK_TILE_BAND
#define NK_TILE_BAND 8
#endif
constexpr uint32_t kTileBand = NK_TILE_BAND;
#ifndef NK_DIRECT_STAGING
#define NK_DIRECT_STAGING 1
#endif
constexpr bool kDirectStaging = NK_DIRECT_STAGING != 0; // A straight into LDS where that applies (see dots_packed_kernel)

struct GemmArgs {
    uint8_t const *a;
    uint8_t const *bp; // packed image (header first)
    uint8_t *c;
    uint64_t a_stride, c_stride, k_src_bytes;
    uint32_t m, n, k;
    uint32_t n_tiles, k_chunks;
    uint32_t tiles_m, tiles_n;
    int avec; // widest load the A pointer and stride allow (1, 2, 4, 8 or 16 bytes)
    int metric; // 0: dot products, 1: angular distances, 2: euclidean distances (kernels built with NORMS)
    union {
        uint32_t chunk_stages; // chunked types: stages between folds of the accumulator (even, 2..16)
        uint32_t strip_waves;  // dots_resident_kernel, which folds every two: wavefronts of a workgroup that have rows
    };
    // Symmetric products (C = A x A^T, upper triangle): only elements with col >= row + tri_shift are stored
    // (`tri_mask` all ones; 0 switches the test off), and the tiles to compute come as a list.
    uint32_t tri_shift, tri_mask;
    // Store-bound shapes: workgroup b starts b * stagger_ticks / gridDim.x ticks of the 100 MHz clock late, so that the
    // compute phases of some compute units fall into the store phases of others (0: all start together).
    union {
        uint32_t stagger_ticks;
        uint32_t strip_tiles; // dots_strips_kernel, which starts its workgroups together: tiles that one walks along a strip (tiles_n counts strips)
    };
    uint32_t store_policy; // 0: by the alignment of C's rows; 1: past the caches; 2: through them
    uint32_t tile_count;       // tiles_m * tiles_n, or the length of the list
    uint32_t const *tile_list; // (tile row, tile column) pairs in walking order, or NULL for the full grid
};
// One more word makes the kernels' argument segments 384 bytes (376 with what the runtime adds), and every launch of every product
// slower, measured with the same code in all else (us): i8 1 x 10,000 x 256 3.67 and 3.84, 2048^3 12.3 and 12.65, 13.05 where
// launches go round three sets of operands.
static_assert(sizeof(GemmArgs) <= 120, "kernel arguments: see above");

/** A triangular grid's tile list (see write_tile_list): up to two launches, `bands` of 8 tile rows each. */
struct TriangleGrid {
    uint32_t tiles_m, tiles_n, bm_log2, bn_log2, shift, bands;
    uint32_t *list;
};
struct TriangleGrids {
    uint32_t pack_blocks; // workgroups of the launch that pack
    TriangleGrid grid[2];
};

/** Scratch memory of a triangular grid, where its tile lists go. `plan`: nothing is launched, the lists that the launch will
 *  read are described there instead. `self`: A is the image's own vectors, from its first on. */
struct TriangleScratch {
    uint32_t *words;
    size_t bytes;
    TriangleGrids *plan;
    bool self;
};

/** The product (or its triangular form) for one element type: picks the tile shape and launches. Defined in
 *  dots_gfx950_<T>.hip. */
hipError_t launch_i8(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_u8(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_bf16(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_f16(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_e4m3(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_e5m2(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_e2m3(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_e2m3_deep(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_e3m2(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_i4(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_u4(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);
hipError_t launch_u1(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle);

/** The wide types (f32, f64; f64 results), dots_gfx950_wide.hip: image = header + k-major f64 with zero padding. */
struct WideGeometry {
    uint32_t elem_bytes, n, k, n_padded, k_padded;
    uint64_t total_bytes;
};
bool wide_geometry(int dtype, size_t n, size_t k, WideGeometry &g);
hipError_t wide_pack(int dtype, void const *b, size_t n, size_t k, size_t b_stride, void *b_packed, hipStream_t stream);
/** `triangle`: only the outputs with col >= row + shift (the symmetric kinds). `metric`: 0 dot products, 1 angular,
 *  2 euclidean distances. */
hipError_t wide_product(int dtype, void const *a, void const *b_packed, void *c, size_t m, size_t n, size_t k,
                        size_t a_stride, size_t c_stride, hipStream_t stream, bool triangle, uint32_t shift, int metric);

/** A fresh non-zero number for the header of a newly packed image. */
uint64_t next_image_nonce();
/** Tile shape forced by nk_hip_set_tile_config for the calling thread (0: the heuristic picks). */
int forced_tile_config();
/** What a call would run as (test hook nk_hip_planned_tile): with the sign bit of forced_tile_config() set, calls are written down
 *  here and not launched. */
struct PlannedTile {
    uint32_t shape, store_policy, units, strip_tiles;
    uint32_t resident_rows, resident_units, resident_tiles; // A in registers instead (nk_hip_planned_resident; rows 0: not)
    uint32_t direct;                                        // A straight into LDS (nk_hip_planned_direct)
};
PlannedTile *planned_tile();
/** Compute units of the current device, asked once per process. */
int compute_unit_count();

} // namespace nk_gfx950

namespace {

using namespace nk_gfx950;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef long v2l __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// nk_dtype_t codes (reference: include/numkong/types.h:923-952)
enum : int {
    kI8 = 1 << 2,
    kU8 = 1 << 6,
    kF16 = 1 << 12,
    kBF16 = 1 << 13,
    kE4M3 = 1 << 14,
    kE5M2 = 1 << 15,
    kI4 = 1 << 16, // two 4-bit integers per byte, the even dimension in the low nibble
    kU4 = 1 << 17,
    kE2M3 = 1 << 18, // 6-bit floats, one per byte (bits 6 and 7 ignored)
    kE3M2 = 1 << 19,
    kU1 = 1 << 1, // eight 1-bit values per byte
    kF64 = 1 << 10, // the two wide types: f64 results, a vector kernel of their own (dots_gfx950_wide.hip)
    kF32 = 1 << 11,
};

constexpr uint32_t kMagic = 0x35394B4Eu; // "NK95"
constexpr uint32_t kVersion = 4;
constexpr int kChunkBytes = 16;   // bytes of K per lane per operand load
constexpr int kTileRows = 32;     // B rows per tile = MFMA N
constexpr int kStageChunks = 8;   // chunks of K per pipeline stage (128 bytes per row)
constexpr int kStageBytes = kStageChunks * kChunkBytes;
constexpr int kTileChunkBytes = kTileRows * kChunkBytes; // 512: one chunk of all 32 rows of a tile

struct PackedHeader {
    uint32_t magic;
    uint32_t version;
    uint32_t dtype;
    uint32_t elem_bytes; // bytes per element as stored in the image (2 for fp8, which is widened to f16)
    uint32_t n;        // logical rows of B = columns of C
    uint32_t k;        // logical depth in elements
    uint32_t n_tiles;  // ceil(n / 32)
    uint32_t k_chunks; // padded depth in 16-byte chunks, multiple of 8
    uint64_t nonce; // a number no other pack call of this process (and, in practice, of any) has used; 0: none
    uint64_t sums_offset; // u32 x (32 * n_tiles): 128 * sum(b') per column for u8, zeros otherwise
    uint64_t total_bytes;
    uint64_t norms_offset; // u32 or f32 x (32 * n_tiles): sum(b^2) per column (exact mod 2^32 for the integer types)
};
static_assert(sizeof(PackedHeader) == 64, "header must stay 64 bytes");

struct Geometry {
    uint32_t elem_bytes;   // bytes per element in the caller's A and B (1 for the 4-bit types, two to a byte)
    uint32_t packed_bytes; // bytes per element in the image and in LDS (fp8 is widened to f16; 0 for bits)
    uint32_t n, k, n_tiles, k_chunks;
    uint64_t k_src_bytes;  // bytes of one source row
    uint64_t data_bytes, sums_bytes, norms_bytes, total_bytes;
};

/** Bits per element in the caller's A and B (0: not a type of this backend). */
inline int elem_bits_of(int dtype) {
    switch (dtype) {
    case kU1: return 1;
    case kI4:
    case kU4: return 4;
    case kI8:
    case kU8:
    case kE4M3:
    case kE5M2:
    case kE2M3:
    case kE3M2: return 8;
    case kF16:
    case kBF16: return 16;
    default: return 0;
    }
}

/** The fp8 MFMA forms of gfx950 align the products inside one lane's k-group to the largest of them and
 *  keep only about 14 bits (1 + 2^-14 comes back as 1), far from the f32 accumulation of the reference's
 *  kernels (dot/serial.h:522-600). e4m3 and e5m2 are therefore widened, exactly, to f16 and run on the f16
 *  MFMA, whose products and sums are kept to full f32 precision: B at pack time, A on its way into LDS.
 *  e3m2 goes the same way (every e3m2 value is an f16 value). e2m3 values are multiples of 1/8 below 8 in magnitude:
 *  eight times each is an i8 value, and the i8 MFMA sums their products exactly at twice the f16 rate, as long as the
 *  i32 sums of 64 x the products cannot overflow (60 * 60 * k < 2^31); deeper rows take the f16 route like e3m2. The
 *  4-bit integers are widened to i8 as well. Single bits stay bits in the image (sixteen to a chunk) and become i8
 *  zeros and ones in registers, on both sides, right in front of the MFMA (their dot product is the popcount of the AND). */
constexpr uint64_t kE2M3IntegerDepth = 0x7FFFFFFFull / 3600; // deepest e2m3 row whose i32 sums are safe
inline bool e2m3_as_integers(size_t k) { return k <= kE2M3IntegerDepth; }

/** Bytes per element in the image and in LDS (0: sub-byte, the 1-bit type). */
inline int packed_bytes_of(int dtype, size_t k) {
    switch (dtype) {
    case kE4M3:
    case kE5M2:
    case kE3M2: return 2;
    case kE2M3: return e2m3_as_integers(k) ? 1 : 2; // (as i8 values, eight times the e2m3 value; or as f16)
    case kI4:
    case kU4: return 1;
    case kU1: return 0;
    default: return elem_bits_of(dtype) / 8;
    }
}
/** Source bytes of a row behind one chunk of the image (a chunk is what one lane feeds one MFMA: 16 bytes of operand). */
inline int source_chunk_of(int dtype, size_t k) {
    switch (dtype) {
    case kE4M3:
    case kE5M2:
    case kE3M2:
    case kI4:
    case kU4: return 8;
    case kE2M3: return e2m3_as_integers(k) ? 16 : 8;
    case kU1: return 2;
    default: return 16;
    }
}
/** Bytes a chunk takes in the image: the 16 operand bytes, except for the 1-bit type, which keeps its 16 bits. */
inline int image_chunk_of(int dtype) { return dtype == kU1 ? 2 : kChunkBytes; }

inline bool make_geometry(int dtype, size_t n, size_t k, Geometry &g) {
    int const bits = elem_bits_of(dtype);
    if (!bits) return false;
    if (n > 0x7FFFFFFFull || k > 0x3FFFFFFFull) return false;
    g.elem_bytes = (uint32_t)(bits + 7) / 8, g.packed_bytes = (uint32_t)packed_bytes_of(dtype, k), g.n = (uint32_t)n, g.k = (uint32_t)k;
    g.k_src_bytes = ((uint64_t)k * bits + 7) / 8; // (sub-byte types: whole bytes, as the reference loads them, cast/serial.h:519-538)
    uint64_t const source_chunk = (uint64_t)source_chunk_of(dtype, k);
    uint64_t const chunks = (g.k_src_bytes + source_chunk - 1) / source_chunk;
    g.k_chunks = (uint32_t)((chunks + 2 * kStageChunks - 1) / (2 * kStageChunks) * (2 * kStageChunks)); // an even number of stages
    g.n_tiles = (uint32_t)((n + kTileRows - 1) / kTileRows);
    g.data_bytes = (uint64_t)g.n_tiles * g.k_chunks * kTileRows * image_chunk_of(dtype);
    g.sums_bytes = (uint64_t)g.n_tiles * kTileRows * sizeof(uint32_t);
    g.norms_bytes = g.sums_bytes;
    g.total_bytes = sizeof(PackedHeader) + g.data_bytes + g.sums_bytes + g.norms_bytes;
    return true;
}


/**
 *  Load one chunk of BYTES (16, 8 or 2) bytes at any address, of which only the first `valid` bytes exist (valid may be
 *  <= 0 or >= BYTES). Missing bytes read as zero; `xr` (0 or 0x80808080) is applied to existing bytes only, so zero
 *  padding stays zero for u8. The aligned dwords that hold the bytes are loaded (each holds one that exists at least, so
 *  nothing outside the matrix's own dwords is touched) and shifted into place, one v_alignbyte_b32 per dword: byte by byte,
 *  a chunk at an odd address took 16 loads.
 */
template <int BYTES>
__device__ __forceinline__ v4i load_chunk_guarded(uint8_t const *p, int valid, uint32_t xr) {
    typedef int v4i_of_dwords __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int kWords = BYTES / 4 > 0 ? BYTES / 4 : 1;
    v4i out = {0, 0, 0, 0};
    if (valid <= 0) return out;
    uint32_t const shift = (uint32_t)(uintptr_t)p & 3u;
    uint32_t const *dwords = (uint32_t const *)(p - shift);
    uint32_t word[kWords + 1];
    if (BYTES == 16 && valid >= BYTES) {
        v4i const wide = *(v4i_of_dwords const *)dwords;
        word[0] = (uint32_t)wide[0], word[1] = (uint32_t)wide[1], word[2] = (uint32_t)wide[2], word[3] = (uint32_t)wide[3];
        word[kWords] = shift ? dwords[4] : 0u;
    }
    else {
#pragma unroll
        for (int w = 0; w <= kWords; ++w) word[w] = 4 * w < (int)shift + (valid < BYTES ? valid : BYTES) ? dwords[w] : 0u;
    }
#pragma unroll
    for (int w = 0; w < kWords; ++w) {
        int const left = valid - 4 * w, bytes = left < 0 ? 0 : (left > 4 ? 4 : left);
        uint32_t const keep = bytes == 4 ? 0xFFFFFFFFu : ((1u << (8 * bytes)) - 1u);
        out[w] = (int)((__builtin_amdgcn_alignbyte(word[w + 1], word[w], shift) ^ xr) & keep);
    }
    if (BYTES < 4) out[0] &= (1 << (8 * (BYTES & 3))) - 1;
    return out;
}

__device__ __forceinline__ uint32_t sum_bytes_u8(v4i v) {
    uint32_t s = __builtin_amdgcn_sad_u8((uint32_t)v[0], 0u, 0u);
    s = __builtin_amdgcn_sad_u8((uint32_t)v[1], 0u, s);
    s = __builtin_amdgcn_sad_u8((uint32_t)v[2], 0u, s);
    s = __builtin_amdgcn_sad_u8((uint32_t)v[3], 0u, s);
    return s;
}

#ifndef NK_E4M3_VIA_BF16
#define NK_E4M3_VIA_BF16 0
#endif
/** e4m3 widened to bf16 and run on the bf16 MFMA instead of f16 (every e4m3 value is a bf16 value as well). Off: on
 *  e4m3 values the two instructions sustain the same rate (MFMA-only loop 1859 against 1848 TFLOP/s) and the product
 *  at 8192^3 takes 0.900 against 0.911 ms, within what two runs differ by, so the image keeps the f16 form. */
constexpr bool kE4M3ViaBF16 = NK_E4M3_VIA_BF16 != 0;

/** Eight OCP fp8 values (two dwords) -> eight f16 values (e4m3 optionally bf16 values), exact for every code incl.
 *  subnormals, Inf, NaN. */
template <bool E5M2>
__device__ __forceinline__ v4i widen_fp8x8(uint32_t lo, uint32_t hi) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    if constexpr (!E5M2 && kE4M3ViaBF16) {
        typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
        v2bf const q0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false), q1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
        v2bf const q2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false), q3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
        v4i wide;
        wide[0] = __builtin_bit_cast(int, q0), wide[1] = __builtin_bit_cast(int, q1);
        wide[2] = __builtin_bit_cast(int, q2), wide[3] = __builtin_bit_cast(int, q3);
        return wide;
    }
    v2h p0, p1, p2, p3;
    if (E5M2) {
        p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(lo, 1.0f, false);
        p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(lo, 1.0f, true);
        p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(hi, 1.0f, false);
        p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(hi, 1.0f, true);
    }
    else {
        p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false);
        p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true);
        p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false);
        p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true);
    }
    v4i out;
    out[0] = __builtin_bit_cast(int, p0), out[1] = __builtin_bit_cast(int, p1);
    out[2] = __builtin_bit_cast(int, p2), out[3] = __builtin_bit_cast(int, p3);
    return out;
}

/**
 *  Eight 6-bit floats, one per byte (two dwords) -> eight f16 values, exact. Both formats are IEEE-like with
 *  subnormals and no Inf/NaN (e2m3: 2 exponent bits, bias 1; e3m2: 3 exponent bits, bias 3; reference decoders:
 *  cast/serial.h:1318-1330, 1455-1470), so the exponent and mantissa bits, moved under an f16's sign bit, read as the
 *  value scaled by a power of two, subnormals included: one packed multiply by 2^14 (e2m3) or 2^12 (e3m2) finishes
 *  two values at a time. Bits 6 and 7 of a byte are ignored, as the reference does. In use for e3m2; e2m3 has the
 *  cheaper integer route of widen_e2m3x4.
 */
template <bool E3M2>
__device__ __forceinline__ v4i widen_fp6x8(uint32_t lo, uint32_t hi) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    constexpr int kShift = E3M2 ? 8 : 7; // exponent field up to bit 10 of the f16
    v2h const scale = E3M2 ? v2h {(_Float16)4096.0f, (_Float16)4096.0f} : v2h {(_Float16)16384.0f, (_Float16)16384.0f};
    v4i out;
#pragma unroll
    for (int pair = 0; pair < 4; ++pair) {
        uint32_t const word = pair < 2 ? lo : hi;
        // bytes 2 * (pair % 2) and 2 * (pair % 2) + 1 of the word, each in a 16-bit lane of its own
        uint32_t const codes = __builtin_amdgcn_perm(0u, word, pair % 2 ? 0x0C030C02u : 0x0C010C00u);
        uint32_t const bits = ((codes << 10) & 0x80008000u) | ((codes & 0x001F001Fu) << kShift);
        v2h const value = __builtin_bit_cast(v2h, bits) * scale;
        out[pair] = __builtin_bit_cast(int, value);
    }
    return out;
}

/**
 *  Four e2m3 values, one per byte -> four i8 values, each EIGHT TIMES the e2m3 value: with 2 exponent bits (bias 1) and
 *  3 mantissa bits every e2m3 value is a multiple of 1/8 of magnitude at most 7.5, so 8 x is an integer in [-60, 60]
 *  (reference decoder: cast/serial.h:1318-1330). Products of two such integers summed in i32 are exact, 64 times the
 *  dot product, and the i8 MFMA runs at twice the rate of the f16 one. All four bytes at once: with x = the low five
 *  bits (e, m), the magnitude is x for e <= 1 (m, or 8 + m), x + (x & 15) for e = 2 (16 + 2 m) and
 *  x + (x & 15) + 2 (x & 7) for e = 3 (32 + 4 m); no byte ever carries into its neighbour. The three per-byte masks
 *  (the two above and 0xFF for a set sign bit) come from 8-entry byte tables indexed by bits 3..5 of each byte, one
 *  v_perm_b32 each. Negative values by 0x80 - magnitude, flipped back. Bits 6 and 7 of a byte are ignored, as the
 *  reference does.
 */
__device__ __forceinline__ uint32_t widen_e2m3x4(uint32_t codes) {
    uint32_t const index = (codes >> 3) & 0x07070707u; // e + 4 * sign, per byte
    uint32_t const negate = __builtin_amdgcn_perm(0xFFFFFFFFu, 0x00000000u, index);  // 0xFF where the sign bit is set
    uint32_t const from_two = __builtin_amdgcn_perm(0x0F0F0000u, 0x0F0F0000u, index); // 0x0F where e >= 2
    uint32_t const at_three = __builtin_amdgcn_perm(0x07000000u, 0x07000000u, index); // 0x07 where e == 3
    uint32_t const low = codes & 0x1F1F1F1Fu;
    uint32_t const magnitude = low + (low & from_two) + ((low & at_three) << 1);
    uint32_t const negative = (0x80808080u - magnitude) ^ 0x80808080u;
    return (negative & negate) | (magnitude & ~negate);
}

/** Sixteen 4-bit integers (two dwords; the even dimension in the low nibble) -> sixteen i8 values: the low nibbles
 *  of a dword's four bytes, then its high nibbles (any order serves as long as A and B use the same one).
 *  Signed: a nibble n with bit 3 set becomes n | 0xF0, the byte-wise (n ^ 8) - 8 of dot/serial.h:781-785. */
template <bool SIGNED>
__device__ __forceinline__ v4i widen_i4x16(uint32_t lo, uint32_t hi) {
    auto extend = [](uint32_t nibbles) {
        if (!SIGNED) return nibbles;
        uint32_t const top = nibbles & 0x08080808u;
        return nibbles | ((top << 5) - (top << 1)); // 0xF0 where bit 3 is set (the last byte's carry leaves the word)
    };
    v4i out;
    out[0] = (int)extend(lo & 0x0F0F0F0Fu), out[1] = (int)extend((lo >> 4) & 0x0F0F0F0Fu);
    out[2] = (int)extend(hi & 0x0F0F0F0Fu), out[3] = (int)extend((hi >> 4) & 0x0F0F0F0Fu);
    return out;
}

/** Sixteen bits (the low half of `bits`, the first dimension in bit 0) -> sixteen i8 values 0 or 1. Four bits times
 *  0x00204081 land in bit 0 of four different bytes. */
__device__ __forceinline__ v4i widen_u1x16(uint32_t bits) {
    v4i out;
#pragma unroll
    for (int w = 0; w < 4; ++w) out[w] = (int)((((bits >> (4 * w)) & 0xFu) * 0x00204081u) & 0x01010101u);
    return out;
}

/** Widening of the source bytes behind one 16-byte chunk, by kind: 1 e4m3, 2 e5m2, 4 e3m2, 8 e2m3 of deep rows (8
 *  bytes to f16); 5 i4, 6 u4 (8 bytes to i8); 7 u1 (2 bytes to i8). Kind 3, e2m3 of rows that are not too deep, turns 16
 *  bytes into 16 i8 values in place (widen_e2m3x4) and does not come through here. */
template <int WIDEN>
__device__ __forceinline__ v4i widen_chunk(uint32_t lo, uint32_t hi) {
    if constexpr (WIDEN == 1) return widen_fp8x8<false>(lo, hi);
    else if constexpr (WIDEN == 2) return widen_fp8x8<true>(lo, hi);
    else if constexpr (WIDEN == 4) return widen_fp6x8<true>(lo, hi);
    else if constexpr (WIDEN == 8) return widen_fp6x8<false>(lo, hi);
    else if constexpr (WIDEN == 5) return widen_i4x16<true>(lo, hi);
    else if constexpr (WIDEN == 6) return widen_i4x16<false>(lo, hi);
    else return widen_u1x16(lo);
}
inline int widen_kind_of(int dtype, size_t k) {
    switch (dtype) {
    case kE4M3: return 1;
    case kE5M2: return 2;
    case kE2M3: return e2m3_as_integers(k) ? 3 : 8;
    case kE3M2: return 4;
    case kI4: return 5;
    case kU4: return 6;
    case kU1: return 7;
    default: return 0;
    }
}

#pragma region Tile lists

/** First tile column of tile row `t` that holds an element on or right of the diagonal col = row + shift; tiles
 *  are 2^bm_log2 rows by 2^bn_log2 columns. */
__host__ __device__ inline uint32_t first_live_tile(uint32_t t, uint32_t bm_log2, uint32_t bn_log2, uint32_t shift) {
    return ((t << bm_log2) + shift) >> bn_log2;
}

/**
 *  The tile list of a triangular grid, in the order of `tile_of_block`: bands of kTileBand tile rows, column
 *  by column within a band, top to bottom within a column, and only tiles with something on or right of the
 *  diagonal. A workgroup writes a band, all of its threads a column at a time. A band's first columns form a staircase (row t
 *  joins at column first_live_tile(t)); the cells left of column c number the sum over its rows of max(0, c -
 *  first_live_tile(t)). Every tile row has a live tile, and a band's rows span whole tiles of columns (kTileBand times
 *  64 rows at least, 512 columns at most), so the bands before this one are an arithmetic series.
 *  The lists are written by the launch that packs the vectors, by workgroups behind its own (a launch of one workgroup in front
 *  of the product took 8 to 11 us of all pairs of 8192, 768 values).
 */
__device__ inline void write_tile_list(TriangleGrids const &grids, uint32_t band) {
    bool const second = band >= grids.grid[0].bands;
    TriangleGrid const &mine = grids.grid[second ? 1 : 0];
    if (second) band -= grids.grid[0].bands;
    uint32_t const tiles_n = mine.tiles_n, first = band * kTileBand, last = first + kTileBand < mine.tiles_m ? first + kTileBand : mine.tiles_m;
    uint32_t joins[kTileBand]; // where each row of the band joins (past the grid for rows that do not exist)
    uint64_t start = 0;
#pragma unroll
    for (uint32_t i = 0; i < kTileBand; ++i) {
        joins[i] = first + i < last ? first_live_tile(first + i, mine.bm_log2, mine.bn_log2, mine.shift) : 0xFFFFFFFFu;
        // (row i of the bands before: `band` of them, each `span` columns of tiles further right than the one above)
        uint32_t const span = (kTileBand << mine.bm_log2) >> mine.bn_log2;
        start += (uint64_t)band * (tiles_n - first_live_tile(i, mine.bm_log2, mine.bn_log2, mine.shift)) - (uint64_t)span * ((uint64_t)band * (band - 1) / 2);
    }
    if (band == 0) start = 0;
    for (uint32_t column = joins[0] + threadIdx.x; column < tiles_n; column += blockDim.x) {
        uint64_t at = start;
#pragma unroll
        for (uint32_t i = 0; i < kTileBand; ++i) at += column > joins[i] ? column - joins[i] : 0;
#pragma unroll
        for (uint32_t i = 0; i < kTileBand; ++i)
            if (joins[i] <= column) mine.list[2 * at] = first + i, mine.list[2 * at + 1] = column, ++at;
    }
}

#pragma endregion Tile lists

#pragma region Packing

/** Sum of the squares of the 8 values of a 16-byte chunk of bf16 (f32 = bits << 16) or f16, in f64. */
template <bool BF16_VALUES>
__device__ __forceinline__ double chunk_sumsq_f64(v4i v) {
    double sum = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float lo, hi;
        if (BF16_VALUES) {
            lo = __builtin_bit_cast(float, (uint32_t)v[w] << 16), hi = __builtin_bit_cast(float, (uint32_t)v[w] & 0xFFFF0000u);
        }
        else {
            typedef _Float16 v2h __attribute__((ext_vector_type(2)));
            int const word = v[w]; // a named copy: bit-casting the vector element expression itself reads element 0
            v2h const pair = __builtin_bit_cast(v2h, word);
            lo = (float)pair[0], hi = (float)pair[1];
        }
        sum = __builtin_fma((double)lo, (double)lo, sum);
        sum = __builtin_fma((double)hi, (double)hi, sum);
    }
    return sum;
}

/**
 *  Packing, one pass: a workgroup of 1024 threads takes one 32-row tile through the whole depth, 32 chunks of every
 *  row per step (thread t: row (t / 8) % 32, chunk 8 * (t / 256) + t % 8 of the step, so 8 neighbouring threads read
 *  128 (64, 16) contiguous source bytes of a row and 8 neighbouring rows write a 128-byte run of the image), and keeps
 *  the per-column terms of what it writes in registers on the way: the u8 compensation term (128 * the sum of the
 *  signed packed bytes of the row, mod 2^32; zero for the other types) and the column's sum of squares, which the
 *  angular and euclidean kinds need (reference: the norms behind the packed rows, dots/serial.h:326-332): exact mod
 *  2^32 for the integer types, accumulated in f64 and rounded once to f32 for the float types. A thread always works
 *  on the same row and on the chunks of one residue mod 32; the 32 partial sums of a row are added in ascending
 *  order of that residue, so the terms do not depend on anything but the row.
 *  WIDEN: 0 copies the elements, 3 rewrites e2m3 bytes as i8 values in place, 7 copies the 16 bits of a chunk of the
 *  1-bit type as they are, otherwise the kind of widen_chunk (8 source bytes per chunk).
 *  KIND, by what the image holds: 0 signed bytes (i8, the widened 4-bit types, e2m3 as 8 x its values), 1 u8 stored
 *  with its offset, 2 bf16, 3 f16 (and what is widened to it), 4 bits (no terms: zeros).
 *  `terms` == 0: the tiles only (callers that will never read the terms). 2: where the byte sums of u8 go, the float types
 *  leave the rows' sums of squares as the loop of the product takes them from A (eight values at a time, in f32): what the
 *  symmetric kinds, which have the image only, need for the bits of the packed ones. (The loop adds the chunks of a stage's
 *  position one after the other; here four threads share them. f64 holds such sums exactly unless the squares span more
 *  than 2^29.)
 *  PAIRS, the symmetric kinds' launch: workgroups past the tiles write the tile lists of a triangular grid (`lists`), a band
 *  each, and `terms` may be 2. A kernel of its own: every workgroup of an ordinary pack would wait for `lists` to be read.
 */
template <int WIDEN, bool BF16_VALUES>
__device__ __forceinline__ double chunk_sumsq_as_staged(v4i v);
constexpr int kPackThreads = 1024;
constexpr int kPackChunks = kPackThreads / kTileRows; // chunks of every row per step of a workgroup
template <int WIDEN, int KIND, bool PAIRS>
__global__ __launch_bounds__(kPackThreads) void pack_kernel(uint8_t const *__restrict__ b, uint64_t b_stride, uint32_t n,
                                                            uint64_t k_src_bytes, uint32_t k_chunks, uint32_t k,
                                                            uint8_t *__restrict__ data, uint32_t *__restrict__ sums,
                                                            uint32_t *__restrict__ norms, int avec, uint32_t xr, int terms,
                                                            PackedHeader header, TriangleGrids lists) {
    if (PAIRS && blockIdx.x >= lists.pack_blocks) return write_tile_list(lists, blockIdx.x - lists.pack_blocks);
    constexpr int kSrcChunk = WIDEN == 0 || WIDEN == 3 ? 16 : (WIDEN == 7 ? 2 : 8);
    constexpr int kImageChunk = WIDEN == 7 ? 2 : kChunkBytes;
    __shared__ int part_sum[kPackChunks][kTileRows];
    __shared__ uint32_t part_squares[kPackChunks][kTileRows];
    __shared__ double part_f64[kPackChunks][kTileRows];
    if (blockIdx.x == 0 && threadIdx.x == 0) *(PackedHeader *)(data - sizeof(PackedHeader)) = header; // (64 bytes in front of the tiles)
    uint32_t const tile = blockIdx.x;
    uint32_t const r = (threadIdx.x >> 3) & 31;
    uint32_t const part = ((threadIdx.x >> 8) << 3) | (threadIdx.x & 7); // chunk of the step = residue of the chunk mod 32
    uint64_t const row = (uint64_t)tile * kTileRows + r;
    uint8_t const *source = b + row * b_stride;
    uint8_t *target = data + ((uint64_t)tile * k_chunks * kTileRows + r) * kImageChunk;
    int sum = 0;
    uint32_t squares = 0;
    double squares_f64 = 0, staged_f64 = 0;
    auto take = [&](uint32_t c) {
        int64_t const left = (int64_t)k_src_bytes - (int64_t)c * kSrcChunk;
        int const valid = row < n ? (int)(left > kSrcChunk ? kSrcChunk : (left < 0 ? 0 : left)) : 0;
        v4i v = {0, 0, 0, 0};
        if (valid > 0) {
            uint8_t const *src = source + (uint64_t)c * kSrcChunk;
            if ((WIDEN == 0 || WIDEN == 3) && valid == 16 && avec >= 16) {
                v = __builtin_nontemporal_load((v4i const *)src); // (read once)
                v[0] ^= (int)xr, v[1] ^= (int)xr, v[2] ^= (int)xr, v[3] ^= (int)xr;
            }
            else { v = load_chunk_guarded<kSrcChunk>(src, valid, xr); }
            if constexpr (WIDEN == 3) {
#pragma unroll
                for (int w = 0; w < 4; ++w) v[w] = (int)widen_e2m3x4((uint32_t)v[w]);
            }
            else if constexpr (WIDEN != 0 && WIDEN != 7) v = widen_chunk<WIDEN>((uint32_t)v[0], (uint32_t)v[1]);
        }
        uint8_t *at = target + (uint64_t)c * (kTileRows * kImageChunk);
        if constexpr (WIDEN == 7) *(uint16_t *)at = (uint16_t)v[0];
        else *(v4i *)at = v;
        if (KIND == 0) {
#pragma unroll
            for (int w = 0; w < 4; ++w) squares = (uint32_t)__builtin_amdgcn_sdot4(v[w], v[w], (int)squares, false);
        }
        else if (KIND == 1) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                sum = __builtin_amdgcn_sdot4(v[w], 0x01010101, sum, false);
                squares = (uint32_t)__builtin_amdgcn_sdot4(v[w], v[w], (int)squares, false);
            }
        }
        else if (KIND == 2 || KIND == 3) {
            squares_f64 += chunk_sumsq_f64<KIND == 2>(v);
            if (PAIRS && terms == 2) staged_f64 += chunk_sumsq_as_staged<WIDEN, KIND == 2>(v);
        }
    };
#pragma unroll 4
    for (uint32_t c = part; c < k_chunks; c += kPackChunks) take(c);
    if (!terms) return;
    part_sum[part][r] = sum, part_squares[part][r] = squares, part_f64[part][r] = squares_f64;
    __syncthreads();
    if (threadIdx.x < kTileRows) {
        uint32_t const mine = threadIdx.x;
        sum = 0, squares = 0, squares_f64 = 0;
#pragma unroll
        for (int p = 0; p < kPackChunks; ++p) sum += part_sum[p][mine], squares += part_squares[p][mine], squares_f64 += part_f64[p][mine];
        // u8 is stored as b - 128 (and its padding as 0): sum(b^2) = sum((b - 128)^2) + 256 * sum(b - 128) + 128^2 * k
        if (KIND == 1) squares += 256u * (uint32_t)sum + 16384u * k;
        sums[(uint64_t)tile * kTileRows + mine] = (uint32_t)sum * 128u;
        norms[(uint64_t)tile * kTileRows + mine] = KIND < 2 ? squares : (KIND == 4 ? 0u : __builtin_bit_cast(uint32_t, (float)squares_f64));
    }
    if (PAIRS && (KIND == 2 || KIND == 3) && terms == 2) {
        __syncthreads();
        part_f64[part][r] = staged_f64;
        __syncthreads();
        if (threadIdx.x < kTileRows) {
            double staged = 0;
#pragma unroll
            for (int position = 0; position < 8; ++position) { // (chunk `position` of every stage, then the positions in turn)
                double one = 0;
#pragma unroll
                for (int p = position; p < kPackChunks; p += 8) one += part_f64[p][threadIdx.x];
                staged += one;
            }
            sums[(uint64_t)tile * kTileRows + threadIdx.x] = __builtin_bit_cast(uint32_t, (float)staged);
        }
    }
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t *p, uint64_t count, uint32_t value) {
    uint64_t const i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) p[i] = value;
}

__global__ __launch_bounds__(64) void write_header_kernel(PackedHeader *dst, PackedHeader h) {
    if (threadIdx.x == 0) *dst = h;
}

/** `tri_mask` all ones: only the elements with col >= row + tri_shift (on or right of a diagonal); 0: all of them. */
__global__ __launch_bounds__(256) void fill_rows_kernel(uint8_t *c, uint32_t m, uint32_t n, uint64_t c_stride,
                                                        uint32_t value, uint32_t tri_shift, uint32_t tri_mask) {
    uint64_t const i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    uint64_t const row = i / n, col = i % n;
    if (row < m && (((uint32_t)row + tri_shift) & tri_mask) <= (uint32_t)col) *(uint32_t *)(c + row * c_stride + col * 4) = value;
}

#pragma endregion Packing

#pragma region Element types

/**
 *  Float accumulation. One MFMA accumulator rounds once per 8 products at the magnitude of the whole running
 *  sum; over a depth of thousands that is 1.4x the error of the reference's scalar kernel for bf16 (4 lanes,
 *  dot/serial.h:406-439), 3x that of its 16-lane AVX-512 kernels (dot/genoa.h:237-256), and 4x the scalar
 *  kernel's for fp8, whose products and short sums are exact in f32 (dot/serial.h:522-600). The float types
 *  therefore fold the accumulator into a second one every `chunk_stages` stages (about an eighth of the depth,
 *  at most 16 stages = 1024 values): the running sums stay short, and the error drops to that of the reference's
 *  best kernels (measured ratios next to the tests). Two accumulator sets do not fit the 256 x 256 tile, so
 *  these types stop at 128 x 256. NK_HALF_SINGLE_ACCUMULATOR builds bf16/f16 without the second set (faster,
 *  less accurate; for comparison only).
 */
#ifdef NK_HALF_SINGLE_ACCUMULATOR
constexpr bool kHalfChunked = false;
#else
constexpr bool kHalfChunked = true;
#endif

struct I8 {
    static constexpr bool kDeepOnly = false; // in use for rows of many stages only
    static constexpr bool kChunked = false; // fold the accumulator into a second one every few stages
    static constexpr int kSrcChunk = 16; // source bytes of A behind one 16-byte LDS chunk
    static constexpr int kImageChunk = kChunkBytes; // bytes of one row's chunk in the image
    static constexpr bool kEightfold = false; // the MFMA sees eight times the values (e2m3 as integers)
    /** What a lane loaded from the image -> its MFMA operand. */
    static __device__ __forceinline__ v4i operand_b(v4i loaded) { return loaded; }
    static __device__ __forceinline__ v4i widen(v4i v) { return v; }
    typedef v16i acc_t;
    typedef uint32_t norm_t; // what a row's sum of squares accumulates in
    static constexpr int kDtype = kI8;
    static constexpr bool kUnsigned = false;
    static constexpr bool kDistances = true; // the distance kinds are built for this type (NORMS kernels)
    static constexpr bool kPrewiden = false; // widen A in place, ahead of its LDS write, spread over two k-steps
    /** Sum of the squares of the source values behind one staged chunk (`raw`: as loaded, `wide`: as it goes to LDS). */
    static __device__ __forceinline__ norm_t sumsq(v4i raw, v4i) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) sum = __builtin_amdgcn_sdot4(raw[w], raw[w], sum, false);
        return (uint32_t)sum;
    }
    static __device__ __forceinline__ void mma(acc_t &acc, v4i a, v4i b) {
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc, 0, 0, 0);
    }
    /** The same with nothing to add to: the first product of a sum (the zero is an operand of the instruction). */
    static __device__ __forceinline__ void mma_fresh(acc_t &acc, v4i a, v4i b) {
        acc_t const zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, zero, 0, 0, 0);
    }
};
struct U8 : I8 {
    static constexpr int kDtype = kU8;
    static constexpr bool kUnsigned = true;
    static __device__ __forceinline__ norm_t sumsq(v4i raw, v4i) {
        uint32_t sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) sum = __builtin_amdgcn_udot4((uint32_t)raw[w], (uint32_t)raw[w], sum, false);
        return sum;
    }
};
struct BF16 {
    static constexpr bool kDeepOnly = false;
    static constexpr bool kChunked = kHalfChunked;
    static constexpr int kSrcChunk = 16; // source bytes of A behind one 16-byte LDS chunk
    static constexpr int kImageChunk = kChunkBytes;
    static constexpr bool kEightfold = false;
    static __device__ __forceinline__ v4i operand_b(v4i loaded) { return loaded; }
    static __device__ __forceinline__ v4i widen(v4i v) { return v; }
    typedef v16f acc_t;
    typedef double norm_t;
    static constexpr int kDtype = kBF16;
    static constexpr bool kUnsigned = false;
    static constexpr bool kDistances = true;
    static constexpr bool kPrewiden = false;
    /** The 8 products are exact in f32; their short sum is rounded a few times, the long sum runs in f64. The short
     *  sum is four `v_dot2_f32_bf16` (two products and the addend each; measured on the part for squares and a
     *  positive addend: within one unit in the last place of the exact sum in 99.3 % of a million cases, 1.43 at
     *  worst), a quarter of the instructions of unpacking to f32 and eight fused multiply-adds. */
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) {
        typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
        float sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            int const word = wide[w]; // a named copy: bit-casting the vector element expression itself reads element 0
            v2bf const pair = __builtin_bit_cast(v2bf, word);
            sum = __builtin_amdgcn_fdot2_f32_bf16(pair, pair, sum, false);
        }
        return (double)sum;
    }
    static __device__ __forceinline__ void mma(acc_t &acc, v4i a, v4i b) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0,
                                                      0, 0);
    }
    static __device__ __forceinline__ void mma_fresh(acc_t &acc, v4i a, v4i b) {
        acc_t const zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), zero, 0,
                                                      0, 0);
    }
};
struct F16 {
    static constexpr bool kDeepOnly = false;
    static constexpr bool kChunked = kHalfChunked;
    static constexpr int kSrcChunk = 16; // source bytes of A behind one 16-byte LDS chunk
    static constexpr int kImageChunk = kChunkBytes;
    static constexpr bool kEightfold = false;
    static __device__ __forceinline__ v4i operand_b(v4i loaded) { return loaded; }
    static __device__ __forceinline__ v4i widen(v4i v) { return v; }
    typedef v16f acc_t;
    typedef double norm_t;
    static constexpr int kDtype = kF16;
    static constexpr bool kUnsigned = false;
    static constexpr bool kDistances = true;
    static constexpr bool kPrewiden = false;
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { // also e4m3 / e5m2, which are f16 by then
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        float sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) { // (mixed-precision fused multiply-adds: `v_dot2_f32_f16` is up to 511 units off for f16 denormals, which e5m2's are)
            int const word = wide[w]; // a named copy: bit-casting the vector element expression itself reads element 0
            v2h const pair = __builtin_bit_cast(v2h, word);
            float const lo = (float)pair[0], hi = (float)pair[1];
            sum = __builtin_fmaf(lo, lo, sum), sum = __builtin_fmaf(hi, hi, sum);
        }
        return (double)sum;
    }
    /** The same short sum with four `v_dot2_f32_f16`, for types whose values are never f16 denormals (measured on
     *  the part for squares of normal numbers and a positive addend: as the bf16 form, 1.44 units at worst). */
    static __device__ __forceinline__ norm_t sumsq_of_normals(v4i wide) {
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        float sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            int const word = wide[w]; // a named copy: bit-casting the vector element expression itself reads element 0
            v2h const pair = __builtin_bit_cast(v2h, word);
            sum = __builtin_amdgcn_fdot2(pair, pair, sum, false);
        }
        return (double)sum;
    }
    static __device__ __forceinline__ void mma(acc_t &acc, v4i a, v4i b) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), acc, 0, 0,
                                                     0);
    }
    static __device__ __forceinline__ void mma_fresh(acc_t &acc, v4i a, v4i b) {
        acc_t const zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), zero, 0, 0,
                                                     0);
    }
};
/** fp8 runs widened to f16 (exact), on the f16 MFMA; see widen_fp8x8. */
struct E4M3 : std::conditional<kE4M3ViaBF16, BF16, F16>::type {
    typedef std::conditional<kE4M3ViaBF16, BF16, F16>::type base_t;
    static constexpr bool kChunked = true;
    static constexpr int kDtype = kE4M3;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_fp8x8<false>((uint32_t)v[0], (uint32_t)v[1]); }
    static __device__ __forceinline__ base_t::norm_t sumsq(v4i raw, v4i wide) {
        if constexpr (kE4M3ViaBF16) return BF16::sumsq(raw, wide);
        else return F16::sumsq_of_normals(wide); // smallest value 2^-9: no f16 denormals
    }
};
struct E5M2 : F16 {
    static constexpr bool kChunked = true;
    static constexpr int kDtype = kE5M2;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_fp8x8<true>((uint32_t)v[0], (uint32_t)v[1]); }
};
/** e2m3 runs as i8 values eight times as large on the i8 MFMA (see widen_e2m3x4): sums are exact integers, 64 times
 *  the dot product, converted to f32 once in the epilogue (one rounding for sums beyond 2^24, none below). */
struct E2M3 : I8 {
    static constexpr int kDtype = kE2M3;
    static constexpr bool kEightfold = true;
    static constexpr bool kPrewiden = true; // 13 operations per dword: too many to sit in front of the LDS writes
    static __device__ __forceinline__ v4i widen(v4i v) {
        v4i out;
#pragma unroll
        for (int w = 0; w < 4; ++w) out[w] = (int)widen_e2m3x4((uint32_t)v[w]);
        return out;
    }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return I8::sumsq(wide, wide); } // 64 x the sum of squares
};
/** e2m3 rows too deep for exact i32 sums (see kE2M3IntegerDepth) run widened to f16 like e3m2: every e2m3 value is an
 *  f16 value, the smallest non-zero one 1/8. */
struct E2M3Deep : F16 {
    static constexpr bool kDeepOnly = true;
    static constexpr bool kChunked = true;
    static constexpr int kDtype = kE2M3;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_fp6x8<false>((uint32_t)v[0], (uint32_t)v[1]); }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return sumsq_of_normals(wide); }
};
/** e3m2 runs widened to f16 (its values times 16 do not fit i8); see widen_fp6x8. */
struct E3M2 : F16 {
    static constexpr bool kChunked = true;
    static constexpr int kDtype = kE3M2;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_fp6x8<true>((uint32_t)v[0], (uint32_t)v[1]); }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return sumsq_of_normals(wide); } // smallest value 2^-4
};
/** The 4-bit integers run widened to i8 on the i8 MFMA; see widen_i4x16. Unsigned nibbles are non-negative i8 values
 *  as they are: none of u8's offset arithmetic. */
struct I4 : I8 {
    static constexpr int kDtype = kI4;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_i4x16<true>((uint32_t)v[0], (uint32_t)v[1]); }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return I8::sumsq(wide, wide); }
};
/** Single bits run as i8 values 0 and 1: sixteen of them behind two source bytes, of A on its way into LDS and of B,
 *  whose image keeps the bits, in registers between the load and the MFMA. */
struct U1 : I8 {
    static constexpr int kDtype = kU1;
    static constexpr bool kDistances = false; // dot products only
    static constexpr int kSrcChunk = 2;
    static constexpr int kImageChunk = 2;
    static __device__ __forceinline__ v4i operand_b(v4i loaded) { return widen_u1x16((uint32_t)loaded[0]); }
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_u1x16((uint32_t)v[0]); }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return I8::sumsq(wide, wide); }
};
struct U4 : I8 {
    static constexpr int kDtype = kU4;
    static constexpr int kSrcChunk = 8;
    static __device__ __forceinline__ v4i widen(v4i v) { return widen_i4x16<false>((uint32_t)v[0], (uint32_t)v[1]); }
    static __device__ __forceinline__ norm_t sumsq(v4i, v4i wide) { return I8::sumsq(wide, wide); }
};

/** Sum of the squares of a chunk as the product's loop takes it (`sumsq` of the type that is stored this way). */
template <int WIDEN, bool BF16_VALUES>
__device__ __forceinline__ double chunk_sumsq_as_staged(v4i v) {
    if constexpr (BF16_VALUES) return BF16::sumsq(v, v);
    else if constexpr (WIDEN == 1 || WIDEN == 4 || WIDEN == 8) return F16::sumsq_of_normals(v);
    else return F16::sumsq(v, v);
}

/**
 *  Distances from a dot product and two sums of squares, as the reference's scalar finalisers compute them
 *  (spatial/serial.h:257-344): integer inputs are converted to f32 first (the i8 kernels read both norms as
 *  signed 32-bit integers, the u8 kernels as unsigned); angular = max(1 - dot * rsqrt(qn * tn), 0), and 0 or
 *  1 when the product of the norms is not positive; euclidean = sqrt(max(qn + tn - 2 * dot, 0)).
 */
template <class T>
__device__ __forceinline__ float norm_as_f32(uint32_t bits) {
    if (T::kDtype == kI8 || T::kDtype == kI4) return (float)(int)bits;
    if (T::kDtype == kU8 || T::kDtype == kU4) return (float)bits;
    if (T::kEightfold) return (float)bits * 0.015625f; // integer sums of squares of 8 x the values
    return __builtin_bit_cast(float, bits);
}

/** What the accumulators hold -> what the caller gets, as 32-bit patterns: as they are, except that e2m3 sums are
 *  integers, 64 times the f32 result. */
template <class T>
__device__ __forceinline__ uint32_t finished_dot(uint32_t bits) {
    if (T::kEightfold) return __builtin_bit_cast(uint32_t, (float)(int)bits * 0.015625f);
    return bits;
}

/** METRIC: 1 angular, 2 euclidean. `query` and `target` are the row's and the column's sums of squares as f32
 *  (converted once per row and once per column of a tile). The reciprocal square root is the hardware's estimate
 *  (1 ulp) refined by one Newton step with fused residuals: identical rows must cancel to within a rounding or
 *  two, as the reference's three Newton steps do (splitting it into a factor per row and a factor per column
 *  would save half of the operations and lose exactly that). */
template <class T, int METRIC>
__device__ __forceinline__ uint32_t distance_from_dot(uint32_t dot_bits, float query, float target) {
    float const dot = T::kDtype == kI8 || T::kDtype == kI4
                          ? (float)(int)dot_bits
                          : (T::kDtype == kU8 || T::kDtype == kU4 ? (float)dot_bits : __builtin_bit_cast(float, dot_bits));
    float result;
    if (METRIC == 1) {
        float const product = query * target;
        float root = __builtin_amdgcn_rsqf(product);
        float const residual = __builtin_fmaf(-(product * root), root, 1.0f);
        root = __builtin_fmaf(root * 0.5f, residual, root);
        float unclipped = __builtin_fmaxf(__builtin_fmaf(-dot, root, 1.0f), 0.0f);
        // Where the dot product squared is the product of the norms exactly (one non-zero term, values of a few bits),
        // a division by a correctly rounded square root gives a cosine of exactly 1 or -1, and so does this.
        if (__builtin_fmaf(dot, dot, -product) == 0.0f) unclipped = dot > 0 ? 0.0f : 2.0f;
        result = product > 0 ? unclipped : (dot == 0 ? 0.0f : 1.0f);
    }
    else {
        // The hardware's reciprocal square root is good to about one unit in the last place; one Newton step on
        // the root itself (residual by a fused multiply-add) leaves it correctly rounded but for rare ties, as
        // the square roots of the reference's vector kernels are.
        float const squared = __builtin_fmaf(-2.0f, dot, query + target);
        float const inverse = __builtin_amdgcn_rsqf(squared);
        float root = squared * inverse;
        root = __builtin_fmaf(__builtin_fmaf(-root, root, squared), 0.5f * inverse, root);
        result = squared > 0 ? root : 0.0f;
    }
    return __builtin_bit_cast(uint32_t, result);
}

/** The hardware's reciprocal square root (good to about a unit in the last place) refined by one Newton step with a
 *  fused residual. Zero gives NaN (infinity times zero), which is what angular_from_factors wants of it. */
__device__ __forceinline__ float refined_rsqrt(float x) {
    float const root = __builtin_amdgcn_rsqf(x);
    float const residual = __builtin_fmaf(-(x * root), root, 1.0f);
    return __builtin_fmaf(root * 0.5f, residual, root);
}

/**
 *  The angular distance where it is cheap: 1 - dot * (rq * rt), with rq and rt the refined reciprocal square roots of
 *  the row's and the column's sums of squares, taken once per row and once per column of a tile instead of once per
 *  output. Three roundings of relative size 2^-24 enter the cosine instead of the one and a half of the full
 *  finaliser, so the form is only used where the cosine is at most a quarter in magnitude (`*cheap`): its error is
 *  then under a unit of 2^-24, below the rounding of the result itself (1 - cos lies in [0.75, 1.25] there). Zero or
 *  overflowed sums of squares make the factors NaN or infinite and fail the test. Everything else, identical rows
 *  above all, takes distance_from_dot.
 */
template <class T>
__device__ __forceinline__ float angular_from_factors(uint32_t dot_bits, float row_factor, float column_factor, bool *cheap) {
    float const dot = T::kDtype == kI8 || T::kDtype == kI4
                          ? (float)(int)dot_bits
                          : (T::kDtype == kU8 || T::kDtype == kU4 ? (float)dot_bits : __builtin_bit_cast(float, dot_bits));
    float const scale = row_factor * column_factor;
    *cheap = __builtin_fabsf(dot * scale) <= 0.25f; // (false for NaN)
    return __builtin_fmaf(-dot, scale, 1.0f);
}

#pragma endregion Element types

#pragma region Packed product

template <int V>
struct slot_c {
    static constexpr int value = V;
};

/** Second-level accumulators: real for the chunked types, empty (no registers) for the others. */
template <class acc_t, int TM, int TN, bool kChunked>
struct Totals {
    acc_t value[TM][TN];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) value[i][j][v] = 0;
    }
    __device__ __forceinline__ void fold(acc_t (&acc)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                value[i][j] += acc[i][j];
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
            }
    }
    __device__ __forceinline__ void clear_block(int i, int j) {
#pragma unroll
        for (int v = 0; v < 16; ++v) value[i][j][v] = 0;
    }
    /** A block's running sum into its total; the sum is left as it is (the next product starts it from zero). */
    __device__ __forceinline__ void fold_block(acc_t const (&acc)[TM][TN], int i, int j) { value[i][j] += acc[i][j]; }
    __device__ __forceinline__ auto finish(acc_t const (&acc)[TM][TN], int i, int j, int v) const {
        return acc[i][j][v] + value[i][j][v];
    }
};
template <class acc_t, int TM, int TN>
struct Totals<acc_t, TM, TN, false> {
    __device__ __forceinline__ void clear() {}
    __device__ __forceinline__ void fold(acc_t (&)[TM][TN]) {}
    __device__ __forceinline__ void clear_block(int, int) {}
    __device__ __forceinline__ void fold_block(acc_t const (&)[TM][TN], int, int) {}
    __device__ __forceinline__ auto finish(acc_t const (&acc)[TM][TN], int i, int j, int v) const { return acc[i][j][v]; }
};


/**
 *  Workgroup index -> output tile. Consecutive workgroup ids are dealt round-robin to the 8 XCDs, each
 *  with a private L2, so ids are first regrouped into 8 contiguous ranges (one per XCD) and each range
 *  walks the tile grid in column-major bands of 8 tile rows: tiles resident on one XCD at the same time
 *  share A row blocks and B column tiles in that XCD's L2.
 *  FEW_ROWS: tiles of 32 rows, which are hardly ever more than one row of tiles and then share nothing but A. All XCDs walk that side by
 *  side, from the image's end to its start: of an image that was packed a moment ago the end is what the last-level cache still holds (us: packed and
 *  multiplied by 16 rows, i8 1,048,576 x 768, 504.6 and 493.7; the product alone 180 and 175, angular bf16 32 x 262,144 x 768 95.3
 *  and 93.9). Not the taller tiles, where the choice costs registers (e2m3 of two stages a workgroup per compute unit: all pairs of 8192 x 219
 *  53.3 and 56.3).
 */
template <bool FEW_ROWS = false>
__device__ __forceinline__ void tile_of_block(uint32_t pid, GemmArgs const &g, uint32_t &tm, uint32_t &tn) {
    uint32_t const tiles_m = g.tiles_m, tiles_n = g.tiles_n;
    uint32_t const total = g.tile_count;
    if (FEW_ROWS && tiles_m == 1) {
        tm = 0, tn = total - 1 - pid;
        return;
    }
    uint32_t const per_xcd = total / 8;
    uint32_t lid = pid;
    if (pid < per_xcd * 8) lid = (pid % 8) * per_xcd + pid / 8;
    if (g.tile_list) { // a triangular grid: the same walk with the tiles left of the diagonal left out, listed
        typedef __attribute__((address_space(4))) uint32_t const constant_u32_t;
        constant_u32_t *entry = (constant_u32_t *)g.tile_list + 2 * (uint64_t)lid;
        tm = entry[0], tn = entry[1];
        return;
    }
    constexpr uint32_t kBand = kTileBand;
    uint32_t const width = kBand * tiles_n;
    uint32_t const band = lid / width;
    uint32_t const first = band * kBand;
    uint32_t const rows = tiles_m - first < kBand ? tiles_m - first : kBand;
    uint32_t const in_band = lid % width;
    tm = first + in_band % rows;
    tn = in_band / rows;
}

/**
 *  A persistent workgroup of 4 wavefronts (one per SIMD) walks over (32*TM) x (128*TN) tiles of C. Every
 *  wavefront owns all 32*TM rows of the tile and its own 32*TN columns: B fragments are loaded by exactly
 *  one wavefront, straight from the packed image into registers; the shared A block goes through LDS.
 *  Being persistent lets the stores of one tile drain while the next tile is already being computed.
 *
 *  A stage is 128 bytes of (packed-width) K per row = four MFMA k-steps. LDS holds two stages of A, rows
 *  128 bytes apart, the 16-byte chunk `c` of row `r` stored at chunk position c ^ ((r >> 1) & 7): the 16
 *  rows that one pass of a ds_read_b128 touches then fall into 16 different 16-byte bank groups (measured:
 *  SQ_LDS_BANK_CONFLICT = 0).
 *
 *  The steady-state loop handles two stages per trip so that every register slot and LDS buffer has a
 *  compile-time index, and its body is one basic block (no branches: prefetch indices are clamped instead),
 *  which keeps the compiler's s_waitcnt counting exact. Everything is fetched two stages ahead:
 *      k-step q MFMAs of (s, q) under the LDS reads of the A fragments of (s, q+1); then the B registers
 *               just consumed are refilled with B(s+2, q)
 *      k-step 2 also moves A(s+1), loaded two stages ago, from registers into the other LDS buffer and
 *               refills those registers with A(s+3)
 *      before the last k-step: one barrier; the first fragments of stage s+1 are read under its MFMAs
 *  The packed image pads K with zeros to an even number of stages; on the A side, the bytes a stage reads
 *  past the end of a row (the next row's, or nothing past the end of the matrix) are masked to zero on their
 *  way into LDS, so ragged depths run through the same loop, and so do rows at any byte address (SHIFTED, below).
 *  Only such rows of fewer than four stages take a plain guarded loop instead.
 *
 *  A is the MFMA's first operand, so a lane ends up with one column and 16 rows of each 32x32 block and the
 *  epilogue stores dwords that are contiguous across lanes: 128 bytes per row per instruction, any C
 *  alignment. (The other orientation, one row and runs of 4 columns per lane stored as 128-bit vectors,
 *  needs a quarter of the store instructions but writes 32-byte pieces of 32 different rows; it measured
 *  12 % slower on the square shapes and 9 % slower on the retrieval shape.)
 */
/** Does a row of A stop short inside a stage's reads, or does the kernel read one stage more than the rows hold (the
 *  image's depth is padded to an even number of stages)? The types whose arithmetic cares (tail_matters_for) clear such
 *  bytes on their way into LDS; kernels compiled with WHOLE are for depths that fill an even number of stages exactly
 *  and leave those masks out of the loop. */
template <class T, bool NORMS>
constexpr bool tail_matters_for() {
    // floats (the image's zero padding times a NaN is a NaN), u8's row sums, the sums of squares of the distances;
    // the integer products need no care: whatever is read there meets zeros of the image
    return NORMS || T::kUnsigned || !__is_same(typename T::acc_t, v16i);
}

/** 16 bytes per lane from a buffer straight into LDS at `dst` + 16 x lane (`dst` the same in all lanes). A function of
 *  its own: the host pass does not know the instruction, and from inside a lambda of a kernel it would take the kernel's
 *  host side with it. */
typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void fetch_to_lds(__amdgpu_buffer_rsrc_t rsrc, lds_void_t *dst, uint32_t lane_offset, uint32_t offset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, dst, 16, lane_offset, offset, 0, 0);
}

/**
 *  DIRECT: A goes from memory straight into LDS (`buffer_load_dwordx4 ... lds`: 64 lanes x 16 bytes land in 1 KiB of LDS
 *  in lane order, so a lane fetches the chunk that belongs at its position of the swizzled row), not through registers
 *  and `ds_write`. LDS is then a ring of four stages, each an array of its own (the compiler tracks what such a load
 *  writes per array, and only so do the waits for one stage's loads not wait for the next stages' as well); a stage's
 *  loads are issued three stages ahead, and one trip of the loop is four stages. For types that reach LDS as they are
 *  in memory, depths of a whole number of trips, the pipelined kernel across tiles, dot products only (the host
 *  checks).
 *
 *  SELF: all pairs of one set of vectors (windows that start on a tile of the image): A is read out of the packed image as well.
 *  There it lies in the order of the operands, widened, with zeros behind the rows' ends and its sums taken, so that
 *  staging is a load and an LDS write of 16 bytes whatever the type, the depth and the alignment of the vectors. Whole calls, before
 *  and now (us), with the tile lists written by the launch that packs: bf16 8192 x 768 angular 134 and 98, 8192 x 4096 417 and 337,
 *  i8 8192 x 768 angular 91 and 75, f16 4096 x 300 dots 53 and 43, e2m3 5000 x 600 euclidean 60 and 48.
 *
 *  SHIFTED: A starts on any byte or its rows are not a multiple of four bytes apart (odd depths). Loads of more than a
 *  dword need dword addresses, so a thread loads the aligned dwords that hold its chunk, one more than the chunk has, and
 *  shifts them into place where they are staged, a v_alignbyte_b32 per dword. How far is the same for every chunk that a
 *  thread stages: its rows are 32 apart, and 32 strides are a multiple of four. Everything behind that (masks, widening,
 *  sums) sees chunks as if A were aligned. Measured against the guarded loop that such rows used to take (whole calls):
 *  i8 3 x 162,699 x 4327 1019 -> 155 us, u8 symmetric 6391 x 7163 1625 -> 252 us, f16 symmetric angular 2947 x 3033
 *  674 -> 113 us; with B packed in the call as well, whose odd rows were read byte by byte: bf16 959 x 74,207 x 4307
 *  6505 -> 1372 us, i8 45 x 610,671 x 391 433 -> 230 us.
 *
 *  FOLDS: the two-accumulator types, depths under 32 stages, where sums go into their totals every two stages, after every
 *  trip of the loop. Then there is no branch around the fold, and no clearing behind it: the next trip's first MFMA of a block
 *  takes a zero operand and stands right behind the 16 additions that empty the block, so that the matrix pipe works on one
 *  block while the next is emptied. With the general form a fold of 128 x 256 results was 256 vector operations between
 *  64 MFMAs. Whole calls, before and now (us): bf16 8192 x 8192 x 1024 184 and 172, 4096 x 4096 x 768 57 and 52, 1000 x 100,000 x
 *  300 263 and 235; e3m2 the same 224 and 193; all pairs of 8192 x 768 119 and 109; the same bits.
 */
// (Workgroups per compute unit: two of 128 x 128 also with two accumulator sets; left to one, the compiler takes 300 registers. The kernels of
// dots on rows at dwords, four stages or more, and those of all pairs need 232 to 255 for that. The others spill: of the 16-bit floats
// distances 6 to 11 registers, 21 on shifted rows, dots on those 2 to 5, two stages 17 and 28; of the 8-bit ones 3 to 8 for distances on
// shifted rows or of two stages. Two are faster all the same: bf16 angular 1024 x 262,144 x 768 768 us through 64 x 128, the best before, and
// 684; distances of 17 to 60 stages, 3000 shapes, 64 x 128 1.10 and 128 x 256 1.26 times the time in the mean, on shifted rows 1.07 to 1.12 and 1.18
// to 1.52 by type.)
template <class T, int TM, int TN, bool ACROSS, bool NORMS = false, bool WHOLE = false, bool DIRECT = false, bool SHIFTED = false, bool FOLDS = false, bool SELF = false>
__global__ __launch_bounds__(256, (TM * TN == 1 ? 4 : TM * TN <= 2 ? 3 : (TM * TN <= 4 ? 2 : 1))) void dots_packed_kernel(GemmArgs g) {
    typedef typename T::acc_t acc_t;
    constexpr int BM = TM * 32;
    constexpr int NT = 256;
    constexpr int kStageLds = BM * kStageBytes;
    constexpr int kLoads = BM * kStageChunks / NT; // 16-byte LDS chunks per thread per stage = TM
    constexpr int kSrcStage = kStageChunks * T::kSrcChunk; // source bytes of A per row per stage
    static_assert(!SELF || (ACROSS && !WHOLE && !DIRECT && !SHIFTED), "A out of the image: only the staged loop has it");
    static_assert(!SHIFTED || (ACROSS && !WHOLE && !DIRECT), "shifted loads: only the staged loop has them");
    static_assert(!DIRECT || (ACROSS && !NORMS && !T::kUnsigned && !T::kPrewiden && T::kSrcChunk == 16 && T::kImageChunk == 16),
                  "straight into LDS: only what needs nothing done to it on the way");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[DIRECT ? 16 : 2 * kStageLds];
    __shared__ __attribute__((aligned(1024))) uint8_t ring0[DIRECT ? kStageLds : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t ring1[DIRECT ? kStageLds : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t ring2[DIRECT ? kStageLds : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t ring3[DIRECT ? kStageLds : 16];
    __shared__ __attribute__((aligned(16))) uint32_t row_terms[T::kUnsigned ? BM : 4]; // u8 only: 128 * (sum of the bytes of each A row of the tile)
    __shared__ uint32_t row_part[T::kUnsigned && !SELF ? 2 * BM * kStageChunks : 1]; // u8 only: the partial sums behind them
    typedef typename T::norm_t norm_t;
    __shared__ __attribute__((aligned(16))) uint32_t row_norms[NORMS ? BM : 4]; // distances only: sum of squares of each A row
    __shared__ __attribute__((aligned(16))) float row_factors[NORMS ? BM : 4];  // ... and its refined reciprocal square root
    __shared__ norm_t norm_part[NORMS && !SELF ? 2 * BM * kStageChunks : 1];              // ... and the partial sums behind them

    uint32_t const tid = threadIdx.x, lane = tid & 63;
    // The wavefront index is the same in all lanes; telling the compiler keeps B addressing in scalar registers.
    uint32_t const wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Trust, but verify: the image must have been packed for this dtype and these dimensions.
    PackedHeader const *header = (PackedHeader const *)g.bp;
    bool const image_ok = header->magic == kMagic && header->version == kVersion &&
                          header->dtype == (uint32_t)T::kDtype && header->n == g.n && header->k == g.k &&
                          header->k_chunks == g.k_chunks && header->n_tiles == g.n_tiles;
    uint8_t const *data = g.bp + sizeof(PackedHeader);
    constexpr int kImageTileChunk = kTileRows * T::kImageChunk; // one chunk of all 32 rows of a tile, as the image holds it
    uint32_t const *col_terms = (uint32_t const *)(data + (uint64_t)g.n_tiles * g.k_chunks * kImageTileChunk);
    uint32_t const *col_norms = col_terms + (uint64_t)g.n_tiles * kTileRows;

    uint32_t const stages = g.k_chunks / kStageChunks;
    // Stages the pipelined loop takes: all of them when A is at least dword-aligned, which is all that multi-dword
    // global loads need, or read by shifted loads; none otherwise. (readfirstlane: the value is uniform, and it must
    // stay in a scalar register because the stage offsets of the buffer loads derive from it.)
    uint32_t const fast = __builtin_amdgcn_readfirstlane(SHIFTED || SELF || g.avec >= (T::kSrcChunk < 4 ? T::kSrcChunk : 4) ? stages : 0);
    uint32_t const xr = T::kUnsigned ? 0x80808080u : 0u;
    uint32_t const a_pos = tid & 7;
    // A fragment reads: lane l takes row l % 32 of each 32-row block and chunk 2q + l / 32.
    uint32_t a_frag[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t const r = lane & 31, c = 2 * q + (lane >> 5);
        a_frag[q] = SELF ? (uint32_t)q * 1024 + lane * 16 : r * kStageBytes + ((c ^ ((r >> 1) & 7)) << 4);
    }

    // A staging: thread t fetches chunk t % 8 of rows i*32 + t/8 of a tile and stores it at its swizzled
    // position. The offsets are the same for every tile: rows past the end of A are cut off by the size of
    // the tile's buffer descriptor (such loads return zeros, and their outputs are never stored).
    uint32_t const a_skew = SHIFTED ? (uint32_t)(uintptr_t)g.a & 3u : 0u; // what the descriptors' bases are rounded down by
    uint32_t const a_shift = SHIFTED ? (a_skew + (tid >> 3) * (uint32_t)g.a_stride + a_pos * T::kSrcChunk) & 3u : 0u;
    uint32_t a_off[kLoads]; // byte offset of the thread's source chunk from the tile's first row
    uint32_t a_lds[kLoads]; // where it goes in an LDS stage
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        uint32_t const r = i * 32 + (tid >> 3);
        a_off[i] = r * (uint32_t)g.a_stride + a_pos * T::kSrcChunk;
        if (SHIFTED) a_off[i] = (a_off[i] + a_skew) & ~3u;
        a_lds[i] = r * kStageBytes + ((a_pos ^ ((r >> 1) & 7)) << 4);
        if (SELF) a_off[i] = i * (g.k_chunks * kImageTileChunk) + tid * T::kImageChunk, a_lds[i] = i * (32 * kStageBytes) + tid * 16;
    }
    uint32_t const b_lane = lane * T::kImageChunk;

    // Loads go through buffer descriptors: one scalar descriptor plus a 32-bit per-lane offset is the cheapest
    // address form to issue (a single address register per lane, no 64-bit vector adds), and a descriptor is
    // all that has to change from one tile to the next. B fragment streams of this wavefront: one descriptor
    // per 32-column tile (tile index clamped to the last one), every lane at offset lane * 16.
    struct TileView {
        uint32_t row0, col0;
        uint8_t const *a; // first row of the tile
        uint32_t a_bytes; // up to the end of its last row that exists
        uint8_t const *b; // first 32-column tile of this wavefront
        uint32_t b_bytes; // up to the end of the packed tiles (or as far as 32 bits reach)
        uint32_t b_tile[TN]; // offsets of the wavefront's tiles from `b`
    };
    auto view_of = [&](uint32_t tile) {
        TileView view;
        uint32_t tile_m, tile_n;
        tile_of_block<TM * TN == 1>(tile, g, tile_m, tile_n);
        view.row0 = tile_m * BM;
        view.col0 = tile_n * (128 * TN) + wave * (32 * TN);
        uint32_t const rows_here = g.m - view.row0 < (uint32_t)BM ? g.m - view.row0 : (uint32_t)BM;
        view.a = g.a + (uint64_t)view.row0 * g.a_stride - a_skew; // (row0 is a multiple of 32: the skew is every tile's)
        // (whole aligned loads: an aligned A never ends in the middle of one that could fault)
        constexpr uint32_t kLoadAlign = T::kSrcChunk < 4 && !SHIFTED ? T::kSrcChunk : 4; // (2-byte loads for the 1-bit type)
        view.a_bytes = SHIFTED ? (a_skew + (rows_here - 1) * (uint32_t)g.a_stride + (uint32_t)g.k_src_bytes + 3u) & ~3u
                               : (rows_here - 1) * (uint32_t)g.a_stride + (((uint32_t)g.k_src_bytes + kLoadAlign - 1) & ~(kLoadAlign - 1));
        uint32_t const tile_bytes = g.k_chunks * kImageTileChunk;
        if constexpr (SELF) { // (rows past the last tile: past the descriptor's end, zeros)
            uint32_t const first_a = (view.row0 + g.tri_shift) / 32;
            uint64_t const left_a = (uint64_t)(g.n_tiles - first_a) * tile_bytes;
            view.a = data + (uint64_t)first_a * tile_bytes, view.a_bytes = left_a < 0xFFFFFFFFull ? (uint32_t)left_a : 0xFFFFFFFFu;
        }
        uint32_t const first = view.col0 / 32 < g.n_tiles ? view.col0 / 32 : g.n_tiles - 1;
        view.b = data + (uint64_t)first * tile_bytes;
        uint64_t const left = (uint64_t)(g.n_tiles - first) * tile_bytes;
        view.b_bytes = left < 0xFFFFFFFFull ? (uint32_t)left : 0xFFFFFFFFu;
#pragma unroll
        for (int j = 0; j < TN; ++j) view.b_tile[j] = (first + j < g.n_tiles ? j : g.n_tiles - 1 - first) * tile_bytes;
        return view;
    };
    auto a_rsrc_of = [](TileView const &view) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)view.a, 0, (int)view.a_bytes, 0x00020000);
    };
    auto b_rsrc_of = [](TileView const &view) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)view.b, 0, (int)view.b_bytes, 0x00020000);
    };

    // When every stage of a tile goes through the pipelined loop, the prefetches of a tile's last stages
    // fetch the first stages of the workgroup's next tile instead of running dry: the pipeline is primed once
    // and then runs across tile boundaries, and the stores of one tile drain under the next tile's MFMAs.
    constexpr bool across = ACROSS; // the host checks that it holds: fast == stages and stages >= 4
    uint32_t const tile_count = g.tile_count;
    // u8 only: every thread sums the unsigned bytes it stages, per staged row, in LDS slots of its own (slot
    // i * 256 + tid: fire-and-forget LDS adds instead of 2 x kLoads registers held through the loop). Two sets:
    // what is staged ahead for the next tile goes to the other one, and the sets swap roles with every tile.
    uint32_t sums_here = 0; // offset of the set of the tile being computed
    if (T::kUnsigned && !SELF) {
#pragma unroll
        for (int i = 0; i < 2 * kLoads; ++i) row_part[i * NT + tid] = 0;
    }
    auto add_row_sum = [&](int i, uint32_t value, uint32_t set) {
        __hip_atomic_fetch_add(&row_part[set + i * NT + tid], value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // Distances: the same bookkeeping for the sums of squares of the rows (u32, or f64 for the float types).
    if (NORMS && !SELF) {
#pragma unroll
        for (int i = 0; i < 2 * kLoads; ++i) norm_part[i * NT + tid] = 0;
    }
    auto add_row_norm = [&](int i, norm_t value, uint32_t set) {
        __hip_atomic_fetch_add(&norm_part[set + i * NT + tid], value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    v4i a_reg[2][kLoads];
    uint32_t a_more[SHIFTED ? 2 : 1][SHIFTED ? kLoads : 1]; // shifted 16-byte chunks: the fifth dword
    v4i b_reg[2][TN][4];
    v4i af[2][TM];

    typedef __attribute__((address_space(1))) uint8_t global_u8_t;
    typedef __attribute__((address_space(1))) uint32_t global_u32_t;
    if (!image_ok) { // the image was not packed for this call: the reference's error convention, all bits set
        for (uint32_t tile = blockIdx.x; tile < g.tile_count; tile += gridDim.x) {
            uint32_t tile_m, tile_n;
            tile_of_block<TM * TN == 1>(tile, g, tile_m, tile_n);
            for (uint32_t at = tid; at < (uint32_t)BM * 128 * TN; at += NT) {
                uint32_t const row = tile_m * BM + at / (128 * TN), col = tile_n * (128 * TN) + at % (128 * TN);
                if (row < g.m && col < g.n && ((row + g.tri_shift) & g.tri_mask) <= col) *(global_u32_t *)((global_u8_t *)g.c + (uint64_t)row * g.c_stride + (uint64_t)col * 4) = 0xFFFFFFFFu;
            }
        }
        return;
    }
    // Persistent workgroups that all start at once stay in step: every compute unit multiplies while none stores,
    // then all of them store at once and share the memory bandwidth, and the two phases add up. Started at evenly
    // spread times instead, some compute while others store, and a shallow product runs at the rate of its stores.
    if (g.stagger_ticks) {
        unsigned long long const until = wall_clock64() + (unsigned long long)blockIdx.x * g.stagger_ticks / gridDim.x;
        while (wall_clock64() < until) __builtin_amdgcn_s_sleep(4);
    }
    TileView cur, nxt;
    acc_t acc[TM][TN];
    constexpr bool kChunked = T::kChunked;
    Totals<acc_t, TM, TN, kChunked> total; // second-level accumulators of the chunked types (see E4M3)

    // A(s) -> registers, in four parts so that the loads can be spread over four k-steps.
    auto load_a = [&](TileView const &view, uint32_t s, auto slot_tag, auto part_tag) {
        constexpr int slot = decltype(slot_tag)::value, part = decltype(part_tag)::value;
        __amdgpu_buffer_rsrc_t const rsrc = a_rsrc_of(view);
        uint32_t const stage_offset = __builtin_amdgcn_readfirstlane(s * (SELF ? kStageChunks * kImageTileChunk : kSrcStage)); // (the same in all lanes: see load_b)
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            if (i * 4 / kLoads != part) continue;
            v4i v = {0, 0, 0, 0};
            if constexpr (SELF) {
                if constexpr (T::kImageChunk == 2) v[0] = (int)(uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, a_off[i], stage_offset, 0);
                else v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, a_off[i], stage_offset, 0));
            }
            else if (T::kSrcChunk == 16) {
                v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, a_off[i], stage_offset, 0));
                if constexpr (SHIFTED) a_more[slot][i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, a_off[i] + 16, stage_offset, 0);
            }
            else if (SHIFTED && T::kSrcChunk == 8) {
                typedef unsigned v3u __attribute__((ext_vector_type(3)));
                v3u const narrow = __builtin_amdgcn_raw_buffer_load_b96(rsrc, a_off[i], stage_offset, 0);
                v[0] = (int)narrow[0], v[1] = (int)narrow[1], v[2] = (int)narrow[2];
            }
            else if (SHIFTED) {
                typedef unsigned v2u __attribute__((ext_vector_type(2)));
                v2u const narrow = __builtin_amdgcn_raw_buffer_load_b64(rsrc, a_off[i], stage_offset, 0);
                v[0] = (int)narrow[0], v[1] = (int)narrow[1];
            }
            else if (T::kSrcChunk == 2) { v[0] = (int)(uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, a_off[i], stage_offset, 0); }
            else {
                typedef unsigned v2u __attribute__((ext_vector_type(2)));
                v2u const narrow = __builtin_amdgcn_raw_buffer_load_b64(rsrc, a_off[i], stage_offset, 0);
                v[0] = (int)narrow[0], v[1] = (int)narrow[1];
            }
            a_reg[slot][i] = v;
        }
    };
    auto load_a_all = [&](TileView const &view, uint32_t s, auto slot_tag) {
        load_a(view, s, slot_tag, slot_c<0>()), load_a(view, s, slot_tag, slot_c<1>());
        load_a(view, s, slot_tag, slot_c<2>()), load_a(view, s, slot_tag, slot_c<3>());
    };
    // Element-wise work on the staged chunks happens here, after the loads have had time to land.
    // `mine` is 1 for a stage of this tile and 0 for one staged ahead for the next tile.
    // `s` is the stage the registers hold: the bytes of its chunk that lie past the end of the row are cleared
    // (for whole stages the masks come out as all ones; no branch either way).
    int const a_tail = (int)(uint32_t)g.k_src_bytes - (int)(a_pos * T::kSrcChunk); // bytes of the row from this thread's chunk on, stage 0
    constexpr bool kMaskTail = !WHOLE && !SELF && tail_matters_for<T, NORMS>();
    constexpr bool kPrewiden = T::kPrewiden && !SELF;
    auto masks_of = [&](uint32_t s, uint32_t (&keep)[(T::kSrcChunk + 3) / 4]) {
        int const left = a_tail - (int)(s * kSrcStage);
#pragma unroll
        for (int w = 0; w < (T::kSrcChunk + 3) / 4; ++w) {
            int const over = left - 4 * w, bytes = over < 0 ? 0 : (over > 4 ? 4 : over);
            keep[w] = bytes == 4 ? 0xFFFFFFFFu : ((1u << (8 * bytes)) - 1u);
        }
    };
    // What a thread loaded for its chunk -> the chunk (SHIFTED; as it is otherwise).
    auto loaded_chunk = [&](auto slot_tag, int i) {
        constexpr int slot = decltype(slot_tag)::value;
        v4i v = a_reg[slot][i];
        if constexpr (SHIFTED) {
            uint32_t const last = T::kSrcChunk == 16 ? a_more[slot][i] : 0u;
#pragma unroll
            for (int w = 0; w < (T::kSrcChunk + 3) / 4; ++w)
                v[w] = (int)__builtin_amdgcn_alignbyte(w < 3 ? (uint32_t)v[w < 3 ? w + 1 : 3] : last, (uint32_t)v[w], a_shift);
        }
        return v;
    };
    // Half of the staged chunks of stage `s`, masked and widened where they are (types with kPrewiden): what
    // store_a would do right in front of its LDS writes, done a k-step or two earlier among that k-step's MFMAs.
    auto prewiden = [&](auto slot_tag, uint32_t s, auto half_tag) {
        constexpr int slot = decltype(slot_tag)::value, half_of = decltype(half_tag)::value;
        constexpr int kSrcWords = (T::kSrcChunk + 3) / 4;
        uint32_t keep[kSrcWords];
        if (kMaskTail) masks_of(s, keep);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            if (i * 2 / kLoads != half_of) continue;
            v4i v = loaded_chunk(slot_tag, i);
            if (kMaskTail) {
#pragma unroll
                for (int w = 0; w < kSrcWords; ++w) v[w] &= (int)keep[w];
            }
            a_reg[slot][i] = T::widen(v);
        }
    };
    auto store_a = [&](auto buffer_tag, auto slot_tag, uint32_t s, uint32_t mine, auto widened_tag) {
        constexpr int buffer = decltype(buffer_tag)::value, slot = decltype(slot_tag)::value;
        constexpr bool widened = decltype(widened_tag)::value != 0; // prewiden has been over these registers
        uint8_t *dst = lds + buffer * kStageLds;
        constexpr int kSrcWords = (T::kSrcChunk + 3) / 4;
        uint32_t keep[kSrcWords];
        if (!widened && kMaskTail) masks_of(s, keep);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            v4i v = widened ? a_reg[slot][i] : loaded_chunk(slot_tag, i);
            if (!widened && kMaskTail) {
#pragma unroll
                for (int w = 0; w < kSrcWords; ++w) v[w] &= (int)keep[w];
            }
            // (without a next tile to stage for, what is staged past the end is dropped)
            uint32_t const set = across && !mine ? sums_here ^ (uint32_t)(kLoads * NT) : sums_here;
            v4i const raw = v;
            if (T::kUnsigned && !SELF) {
                uint32_t const sum = sum_bytes_u8(v);
                add_row_sum(i, across ? sum : sum * mine, set);
                v[0] ^= (int)xr, v[1] ^= (int)xr, v[2] ^= (int)xr, v[3] ^= (int)xr;
            }
            v4i const wide = widened || (SELF && T::kImageChunk == 16) ? v : T::widen(v);
            if (NORMS && !SELF) {
                norm_t const squares = T::sumsq(raw, wide);
                add_row_norm(i, across || mine ? squares : (norm_t)0, set);
            }
            *(v4i *)(dst + a_lds[i]) = wide;
        }
    };
    auto load_b = [&](TileView const &view, uint32_t s, auto slot_tag, auto q_tag) {
        constexpr int slot = decltype(slot_tag)::value, q = decltype(q_tag)::value;
        __amdgpu_buffer_rsrc_t const rsrc = b_rsrc_of(view);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            // (the same in all lanes; saying so keeps the offset a scalar operand where the compiler has lost track of it,
            // instead of a loop over the lanes' values)
            uint32_t const tile_offset = __builtin_amdgcn_readfirstlane(view.b_tile[j] + s * (kStageChunks * kImageTileChunk));
            if constexpr (T::kImageChunk == 2) // (sixteen bits per lane: the rest of the register is never looked at)
                b_reg[slot][j][q][0] = (int)(uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, b_lane + q * 2 * kImageTileChunk, tile_offset, 0);
            else
                b_reg[slot][j][q] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, b_lane + q * 2 * kImageTileChunk, tile_offset, 0));
        }
    };
    auto ring_of = [&](auto index_tag) -> uint8_t * {
        constexpr int index = decltype(index_tag)::value & 3;
        return index == 0 ? ring0 : (index == 1 ? ring1 : (index == 2 ? ring2 : ring3));
    };
    auto read_frags = [&](auto buffer_tag, auto q_tag, auto parity_tag) {
        constexpr int buffer = decltype(buffer_tag)::value, q = decltype(q_tag)::value,
                      parity = decltype(parity_tag)::value;
        uint8_t const *src = (DIRECT ? ring_of(buffer_tag) : lds + buffer * kStageLds) + a_frag[q];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[parity][i] = *(v4i const *)(src + i * 32 * kStageBytes);
    };
    auto multiply = [&](auto slot_tag, auto q_tag) {
        constexpr int slot = decltype(slot_tag)::value, q = decltype(q_tag)::value;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            v4i const b = T::operand_b(b_reg[slot][j][q]);
#pragma unroll
            for (int i = 0; i < TM; ++i) T::mma(acc[i][j], af[q & 1][i], b);
        }
    };
    // The same for the first k-step of a tile: its MFMAs start the sums from a zero operand, so that no accumulator is
    // ever cleared (the totals of the chunked types are, a block's in front of its MFMA).
    auto multiply_fresh = [&](auto slot_tag, auto q_tag, auto fold_tag) {
        constexpr int slot = decltype(slot_tag)::value, q = decltype(q_tag)::value;
        constexpr bool fold = decltype(fold_tag)::value != 0; // in the middle of a tile: the running sum goes into the total
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            v4i const b = T::operand_b(b_reg[slot][j][q]);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if constexpr (fold) total.fold_block(acc, i, j);
                else total.clear_block(i, j);
                T::mma_fresh(acc[i][j], af[q & 1][i], b);
            }
        }
    };
    // What staging one chunk of A costs besides its LDS write: vector operations (u8: four exclusive-ors and the byte
    // sums; the distance kinds: the squares) and LDS adds (one per sum kept). The k-step that stages asks for them
    // behind its MFMAs, a chunk's worth each; left alone they all land between the last MFMA and the barrier.
    constexpr bool kIntegerSums = __is_same(typename T::acc_t, v16i);
    constexpr int kStageVector = SELF ? 0 : (T::kUnsigned ? 8 : 0) + (NORMS ? (kIntegerSums ? 5 : 28) : 0) + (SHIFTED && !T::kPrewiden ? (T::kSrcChunk + 3) / 4 : 0);
    constexpr int kStageLoads = (kLoads >= 4 ? kLoads / 4 : 1) * (SHIFTED && T::kSrcChunk == 16 ? 2 : 1); // of A, per k-step
    constexpr int kStageDs = SELF ? 1 : 1 + (T::kUnsigned ? 1 : 0) + (NORMS ? 1 : 0);
    // Scheduling hints for one k-step. Masks: 0x008 MFMA, 0x020 VMEM read, 0x100 DS read, 0x200 DS write.
    // Fragment reads go one-to-one with the first TM MFMAs; the global loads of the k-step (TN of B
    // and a quarter of A) are spread over the remaining MFMAs; k-step 2 also carries the LDS writes.
    auto schedule_k_step = [&](auto writes_tag, auto vector_tag) {
        constexpr bool writes = decltype(writes_tag)::value != 0;
        constexpr int vector = decltype(vector_tag)::value; // vector operations to put behind every MFMA (0x002)
        constexpr int loads = TN + kStageLoads;
        constexpr int rest = TM * (TN - 1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (vector > 0) __builtin_amdgcn_sched_group_barrier(0x002, vector, 0);
        }
        if constexpr (rest == 0) {
            if (writes) __builtin_amdgcn_sched_group_barrier(0x200, kLoads, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);
        }
        else if constexpr (writes && kStageDs > 1) {
            // The LDS adds are atomics, and the compiler keeps atomics in program order with every other memory
            // operation, this k-step's loads included (which cannot go early anyway: the second half of the MFMAs
            // still reads the registers that B's loads refill). So the stage's k-step 2 stages first in program order,
            // a chunk in front of each MFMA of the second half, and all its loads go behind the last MFMA.
#pragma unroll
            for (int i = 0; i < rest; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if constexpr (vector > 0) __builtin_amdgcn_sched_group_barrier(0x002, vector, 0);
                if (i < kLoads) __builtin_amdgcn_sched_group_barrier(0x080, kStageDs, 0); // (0x080: any LDS operation)
            }
            if (kLoads > rest) __builtin_amdgcn_sched_group_barrier(0x080, kStageDs * (kLoads - rest), 0);
            __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);
        }
        else {
#pragma unroll
            for (int i = 0; i < rest; ++i) {
                if (writes && i < kLoads) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                if (i * loads / rest != (i + 1) * loads / rest || (loads > rest && i == 0))
                    __builtin_amdgcn_sched_group_barrier(0x020, loads > rest ? loads : 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if constexpr (vector > 0) __builtin_amdgcn_sched_group_barrier(0x002, vector, 0);
            }
            if (writes && kLoads > rest) __builtin_amdgcn_sched_group_barrier(0x200, kLoads - rest, 0);
        }
    };
    // The first k-step of a tile of the chunked types: in front of every MFMA the 16 zeros of its block's total;
    // fragment reads and loads as in any k-step without LDS writes.
    auto schedule_fresh_k_step = [&]() {
        constexpr int loads = TN + kStageLoads;
#pragma unroll
        for (int i = 0; i < TM * TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
            if (i < TM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i >= TM && i - TM < loads) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        if (TM * TN - TM < loads) __builtin_amdgcn_sched_group_barrier(0x020, loads - (TM * TN - TM), 0);
    };
    // One stage of the steady state; `P` = stage parity = LDS buffer = register slot. Stages s+2 and
    // s+3 are fetched here; past the tile's end they are the first stages of `nxt` (the next tile, or
    // this one again when nothing follows: loads of valid memory that nobody uses).
    // `inside`: how many of the stages s + 2, s + 3 are known to be this tile's (a tile's first two stages, whose numbers
    // are constants and which the host guarantees two or three more: see stage_direct).
    auto stage = [&](auto parity_tag, uint32_t s, auto entry_tag, auto inside_tag) __attribute__((always_inline)) {
        constexpr int P = decltype(parity_tag)::value;
        constexpr int entry = decltype(entry_tag)::value; // 0: in the middle of a sum; 1: a fold in front of it; 2: the first stage of a tile
        constexpr int inside = ACROSS ? decltype(inside_tag)::value : 0; // (without ACROSS a tile may have two stages only)
        // vector operations behind each MFMA of the k-steps that widen in place: their share of half the chunks
        constexpr int kSpread = kPrewiden ? (kLoads * 28 + TM * TN - 1) / (TM * TN) : 0;
        bool const wrap2 = inside < 1 && s + 2 >= fast, wrap3 = inside < 2 && s + 3 >= fast;
        uint32_t const s2 = wrap2 ? s + 2 - fast : s + 2, s3 = wrap3 ? s + 3 - fast : s + 3;
        TileView const &a2 = wrap2 ? nxt : cur, &a3 = wrap3 ? nxt : cur, &b2 = a2;
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<P>(), slot_c<1>(), slot_c<1>());
        if constexpr (entry != 0) multiply_fresh(slot_c<P>(), slot_c<0>(), slot_c<entry == 1>());
        else multiply(slot_c<P>(), slot_c<0>());
        load_b(b2, s2, slot_c<P>(), slot_c<0>()), load_a(a2, s2, slot_c<P>(), slot_c<2>());
        if constexpr (kPrewiden) prewiden(slot_c<P ^ 1>(), s + 1 < fast ? s + 1 : 0u, slot_c<0>());
        if constexpr (entry != 0 && kChunked) schedule_fresh_k_step();
        else schedule_k_step(slot_c<0>(), slot_c<kSpread>());
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<P>(), slot_c<2>(), slot_c<0>());
        multiply(slot_c<P>(), slot_c<1>());
        load_b(b2, s2, slot_c<P>(), slot_c<1>()), load_a(a2, s2, slot_c<P>(), slot_c<3>());
        if constexpr (kPrewiden) prewiden(slot_c<P ^ 1>(), s + 1 < fast ? s + 1 : 0u, slot_c<1>());
        schedule_k_step(slot_c<0>(), slot_c<kSpread>());
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<P>(), slot_c<3>(), slot_c<1>());
        multiply(slot_c<P>(), slot_c<2>());
        if constexpr (kStageDs == 1) load_b(b2, s2, slot_c<P>(), slot_c<2>());
        // A(s+1), loaded over the last two stages, goes to the other buffer (every wavefront left it
        // at the previous barrier); then its registers start being refilled with A(s+3).
        bool const mine = s + 1 < fast;
        store_a(slot_c<P ^ 1>(), slot_c<P ^ 1>(), mine ? s + 1 : 0u, mine ? 1u : 0u, slot_c<kPrewiden ? 1 : 0>());
        if constexpr (kStageDs > 1) load_b(b2, s2, slot_c<P>(), slot_c<2>()); // (see schedule_k_step)
        load_a(a3, s3, slot_c<P ^ 1>(), slot_c<0>());
        schedule_k_step(slot_c<1>(), slot_c<kStageVector>());
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<P ^ 1>(), slot_c<0>(), slot_c<0>());
        multiply(slot_c<P>(), slot_c<3>());
        load_b(b2, s2, slot_c<P>(), slot_c<3>()), load_a(a3, s3, slot_c<P ^ 1>(), slot_c<1>());
        schedule_k_step(slot_c<0>(), slot_c<0>());
    };

    // ---- A straight into LDS (DIRECT) ----
    // Fetch t of a wavefront brings the 8 rows from 8 * (4 t + wave) on: lane l lands at row l / 8, position l % 8 of
    // the 1 KiB that starts there, so it fetches the chunk that the swizzle puts at that position.
    uint32_t a_direct[DIRECT ? kLoads : 1];
    if constexpr (DIRECT) {
#pragma unroll
        for (int t = 0; t < kLoads; ++t) {
            uint32_t const r = 8 * (4 * t + wave) + (lane >> 3);
            a_direct[t] = r * (uint32_t)g.a_stride + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
        }
    }
    auto fetch_a = [&](TileView const &view, uint32_t s, auto ring_tag, auto part_tag) __attribute__((always_inline)) {
        constexpr int part = decltype(part_tag)::value;
        __amdgpu_buffer_rsrc_t const rsrc = a_rsrc_of(view);
        uint32_t const stage_offset = __builtin_amdgcn_readfirstlane(s * kSrcStage);
        uint8_t *stage_base = ring_of(ring_tag);
#pragma unroll
        for (int t = 0; t < kLoads; ++t) {
            if (t * 4 / kLoads != part) continue;
            fetch_to_lds(rsrc, (lds_void_t *)(stage_base + (4 * t + wave) * 1024), a_direct[DIRECT ? t : 0], stage_offset);
        }
    };
    auto fetch_a_all = [&](TileView const &view, uint32_t s, auto ring_tag) __attribute__((always_inline)) {
        fetch_a(view, s, ring_tag, slot_c<0>()), fetch_a(view, s, ring_tag, slot_c<1>());
        fetch_a(view, s, ring_tag, slot_c<2>()), fetch_a(view, s, ring_tag, slot_c<3>());
    };
    // Every wavefront waits for its own fetches into a stage, then all meet: after that the stage is whole for everybody. `younger`:
    // the fetches and loads that a wavefront has issued behind those, at the least (stores of a tile come on top); memory answers in
    // order. The compiler puts the same wait in front of the word read below, of its own accord, but it has once left such waits out, and
    // then results were wrong now and then: written here, the wait does not depend on it.
    // No fence: a fence would wait for the fetches of the later stages as well. The waits for the fragment reads
    // that are still in flight come with the word read (LDS answers in order).
    auto stage_arrived = [&](auto ring_tag, auto younger_tag) __attribute__((always_inline)) {
        constexpr int younger = decltype(younger_tag)::value;
        static_assert(younger < 64, "what a wait can count to");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70 | (younger & 15) | (younger >> 4) << 14);
        typedef __attribute__((address_space(3))) uint32_t const lds_u32_t;
        uint32_t const word = *(lds_u32_t *)(ring_of(ring_tag) + lane * 4);
        asm volatile("" ::"v"(word) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // One stage: `R` = its place in the ring, `P` = the register slot of its B (stage parity). A(s+3) is fetched into
    // the ring stage that the barrier of the stage before has freed; B(s+2) into the registers just used.
    auto schedule_direct_k_step = [&]() {
        constexpr int loads = TN + (kLoads >= 4 ? kLoads / 4 : 1);
        constexpr int rest = TM * (TN - 1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        if constexpr (rest == 0) __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);
        else {
#pragma unroll
            for (int i = 0; i < rest; ++i) {
                if (i * loads / (rest ? rest : 1) != (i + 1) * loads / (rest ? rest : 1) || (loads > rest && i == 0))
                    __builtin_amdgcn_sched_group_barrier(0x020, loads > rest ? loads : 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
        }
    };
    // (`inside`: stages s + 2 and s + 3 are known to be this tile's, as in a tile's first trip, whose stage numbers are
    // constants: left to choose, the compiler computes the choices once, in vector registers that it then spills, and
    // the reload of a spill is a load whose wait is a wait for everything prefetched)
    auto stage_direct = [&](auto ring_tag, uint32_t s, auto entry_tag, auto inside_tag) __attribute__((always_inline)) {
        constexpr int R = decltype(ring_tag)::value & 3, P = R & 1;
        constexpr int entry = decltype(entry_tag)::value;
        constexpr bool inside = decltype(inside_tag)::value != 0;
        bool const wrap2 = !inside && s + 2 >= fast, wrap3 = !inside && s + 3 >= fast;
        uint32_t const s2 = wrap2 ? s + 2 - fast : s + 2, s3 = wrap3 ? s + 3 - fast : s + 3;
        TileView const &b2 = wrap2 ? nxt : cur, &a3 = wrap3 ? nxt : cur;
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<R>(), slot_c<1>(), slot_c<1>());
        if constexpr (entry != 0) multiply_fresh(slot_c<P>(), slot_c<0>(), slot_c<entry == 1>());
        else multiply(slot_c<P>(), slot_c<0>());
        load_b(b2, s2, slot_c<P>(), slot_c<0>()), fetch_a(a3, s3, slot_c<R + 3>(), slot_c<0>());
        if constexpr (entry != 0 && kChunked) schedule_fresh_k_step();
        else schedule_direct_k_step();
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<R>(), slot_c<2>(), slot_c<0>());
        multiply(slot_c<P>(), slot_c<1>());
        load_b(b2, s2, slot_c<P>(), slot_c<1>()), fetch_a(a3, s3, slot_c<R + 3>(), slot_c<1>());
        schedule_direct_k_step();
        __builtin_amdgcn_sched_barrier(0);
        read_frags(slot_c<R>(), slot_c<3>(), slot_c<1>());
        multiply(slot_c<P>(), slot_c<2>());
        load_b(b2, s2, slot_c<P>(), slot_c<2>()), fetch_a(a3, s3, slot_c<R + 3>(), slot_c<2>());
        schedule_direct_k_step();
        // (behind the fetches of stage s + 1: B and A of the stage before this one, and three quarters of both of this one)
        stage_arrived(slot_c<R + 1>(), slot_c<7 * TN + kLoads + kLoads * 3 / 4>());
        read_frags(slot_c<R + 1>(), slot_c<0>(), slot_c<0>());
        multiply(slot_c<P>(), slot_c<3>());
        load_b(b2, s2, slot_c<P>(), slot_c<3>()), fetch_a(a3, s3, slot_c<R + 3>(), slot_c<3>());
        schedule_direct_k_step();
    };
    auto prime_direct = [&]() {
        __syncthreads();
        fetch_a_all(cur, 0, slot_c<0>());
        load_b(cur, 0, slot_c<0>(), slot_c<0>()), load_b(cur, 0, slot_c<0>(), slot_c<1>());
        load_b(cur, 0, slot_c<0>(), slot_c<2>()), load_b(cur, 0, slot_c<0>(), slot_c<3>());
        fetch_a_all(cur, 1, slot_c<1>());
        load_b(cur, 1, slot_c<1>(), slot_c<0>()), load_b(cur, 1, slot_c<1>(), slot_c<1>());
        load_b(cur, 1, slot_c<1>(), slot_c<2>()), load_b(cur, 1, slot_c<1>(), slot_c<3>());
        fetch_a_all(cur, 2, slot_c<2>());
        stage_arrived(slot_c<0>(), slot_c<8 * TN + 2 * kLoads>());
        read_frags(slot_c<0>(), slot_c<0>(), slot_c<0>());
    };

    // Fills the pipeline for a tile: stages 0 and 1 on their way, A(0) in LDS, its first fragments read.
    auto prime = [&]() {
        __syncthreads(); // the previous tile's last fragment reads are done
        load_a_all(cur, 0, slot_c<0>());
        load_b(cur, 0, slot_c<0>(), slot_c<0>()), load_b(cur, 0, slot_c<0>(), slot_c<1>());
        load_b(cur, 0, slot_c<0>(), slot_c<2>()), load_b(cur, 0, slot_c<0>(), slot_c<3>());
        load_a_all(cur, 1, slot_c<1>());
        load_b(cur, 1, slot_c<1>(), slot_c<0>()), load_b(cur, 1, slot_c<1>(), slot_c<1>());
        load_b(cur, 1, slot_c<1>(), slot_c<2>()), load_b(cur, 1, slot_c<1>(), slot_c<3>());
        store_a(slot_c<0>(), slot_c<0>(), 0u, 1u, slot_c<0>());
        // the first half of A(2), as k-steps 2 and 3 of a stage "-1" would have issued it
        // (with two stages in all it is A(0) again, which nobody uses)
        uint32_t const third = fast > 2 ? 2 : 0;
        load_a(cur, third, slot_c<0>(), slot_c<0>()), load_a(cur, third, slot_c<0>(), slot_c<1>());
        __syncthreads();
        read_frags(slot_c<0>(), slot_c<0>(), slot_c<0>());
    };
    if constexpr (across) {
        cur = view_of(blockIdx.x);
        if constexpr (DIRECT) prime_direct();
        else prime();
    }

    for (uint32_t tile = blockIdx.x; tile < tile_count; tile += gridDim.x) {
        cur = view_of(tile);
        bool const has_next = across && tile + gridDim.x < tile_count;
        nxt = view_of(has_next ? tile + gridDim.x : tile);
        uint32_t const row0 = cur.row0, col0 = cur.col0;

        // u8: the column terms of this tile are fetched now and used in the epilogue, so that nothing has to
        // wait for them (a wait for a load is a wait for every store issued before it).
        uint32_t col_term[TN], col_norm[TN];
        // Vectors with themselves: a row's terms are its column's, but for the sums of squares of the floats, which the pack
        // kernel has left where u8 keeps its byte sums (added up as the loop of a product of two matrices does it).
        uint32_t self_term = 0, self_norm = 0;
        if constexpr (SELF && (T::kUnsigned || NORMS)) {
            uint32_t const row = row0 + g.tri_shift + tid, last = g.n_tiles * kTileRows - 1;
            if (T::kUnsigned) self_term = col_terms[row < last ? row : last] + 16384u * g.k;
            if (NORMS) self_norm = (kIntegerSums ? col_norms : col_terms)[row < last ? row : last];
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            col_term[j] = 0, col_norm[j] = 0;
            uint32_t const t = col0 / 32 + j < g.n_tiles ? col0 / 32 + j : g.n_tiles - 1;
            if constexpr (T::kUnsigned) col_term[j] = col_terms[(uint64_t)t * kTileRows + (lane & 31)];
            if constexpr (NORMS) col_norm[j] = col_norms[(uint64_t)t * kTileRows + (lane & 31)];
        }

        {
            if (across || fast > 0) { // (always, when the pipeline runs across tiles: the host checked)
                if constexpr (!across) prime();
                // Nothing is cleared at the start of a tile: in its first k-step the first MFMA of every block takes a
                // zero operand (and the totals of the chunked types are zeroed next to it). Chunked types: every
                // `chunk_stages` stages the running sums go into the totals.
                uint32_t until_fold = g.chunk_stages;
                auto fold_when_due = [&]() __attribute__((always_inline)) {
                    if constexpr (kChunked) {
                        until_fold -= 2;
                        if (until_fold == 0) {
                            __builtin_amdgcn_sched_barrier(0);
                            total.fold(acc);
                            until_fold = g.chunk_stages;
                        }
                    }
                };
                if constexpr (DIRECT) { // (four stages a trip: the host checked that the depth, and a chunk, are whole trips)
                    auto fold_after_trip = [&]() __attribute__((always_inline)) {
                        if constexpr (kChunked) {
                            until_fold -= 4;
                            if (until_fold == 0) {
                                __builtin_amdgcn_sched_barrier(0);
                                total.fold(acc);
                                until_fold = g.chunk_stages;
                            }
                        }
                    };
                    stage_direct(slot_c<0>(), 0u, slot_c<2>(), slot_c<1>()); // (at least eight stages: the host checked)
                    stage_direct(slot_c<1>(), 1u, slot_c<0>(), slot_c<1>());
                    stage_direct(slot_c<2>(), 2u, slot_c<0>(), slot_c<1>());
                    stage_direct(slot_c<3>(), 3u, slot_c<0>(), slot_c<1>());
                    fold_after_trip();
                    for (uint32_t s = 4; s < fast; s += 4) {
                        stage_direct(slot_c<0>(), s, slot_c<0>(), slot_c<0>());
                        stage_direct(slot_c<1>(), s + 1, slot_c<0>(), slot_c<0>());
                        stage_direct(slot_c<2>(), s + 2, slot_c<0>(), slot_c<0>());
                        stage_direct(slot_c<3>(), s + 3, slot_c<0>(), slot_c<0>());
                        fold_after_trip();
                    }
                }
                else {
                    stage(slot_c<0>(), 0u, slot_c<2>(), slot_c<2>()); // (with ACROSS at least four stages: the host checked)
                    stage(slot_c<1>(), 1u, slot_c<0>(), slot_c<1>());
                    if constexpr (!FOLDS) fold_when_due();
                    for (uint32_t s = 2; s < fast; s += 2) {
                        stage(slot_c<0>(), s, slot_c<FOLDS>(), slot_c<0>());
                        stage(slot_c<1>(), s + 1, slot_c<0>(), slot_c<0>());
                        if constexpr (!FOLDS) fold_when_due();
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }

            // Remaining stages: the ragged end of K, or everything when A cannot be read with vector loads.
            if (!across && fast < stages) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
                total.clear();
                uint8_t const *a_tile = g.a + (uint64_t)row0 * g.a_stride;
                uint32_t a_slow[kLoads]; // rows clamped to the last one: plain loads have no descriptor to stop them
#pragma unroll
                for (int i = 0; i < kLoads; ++i) {
                    uint32_t const r = i * 32 + (tid >> 3);
                    uint32_t const row = row0 + r < g.m ? r : g.m - 1 - row0;
                    a_slow[i] = row * (uint32_t)g.a_stride + a_pos * T::kSrcChunk;
                }
                uint32_t until_fold = g.chunk_stages;
                for (uint32_t s = fast; s < stages; ++s) {
                    __syncthreads();
                    int64_t const left = (int64_t)g.k_src_bytes - (int64_t)s * kSrcStage - (int64_t)a_pos * T::kSrcChunk;
                    int const valid = (int)(left > T::kSrcChunk ? T::kSrcChunk : (left < 0 ? 0 : left));
#pragma unroll
                    for (int i = 0; i < kLoads; ++i) {
                        v4i v = load_chunk_guarded<T::kSrcChunk>(a_tile + (uint64_t)s * kSrcStage + a_slow[i], valid, 0u);
                        v4i const raw = v;
                        if (T::kUnsigned) {
                            add_row_sum(i, sum_bytes_u8(v), sums_here);
#pragma unroll
                            for (int w = 0; w < 4; ++w) { // flip only bytes that exist: the zero padding stays zero
                                int const rem = valid - 4 * w;
                                uint32_t const mask = rem >= 4 ? 0x80808080u : (rem <= 0 ? 0u : (0x80808080u >> (8 * (4 - rem))));
                                v[w] ^= (int)mask;
                            }
                        }
                        v4i const wide = T::widen(v);
                        if (NORMS) add_row_norm(i, T::sumsq(raw, wide), sums_here);
                        *(v4i *)(lds + a_lds[i]) = wide;
                    }
                    load_b(cur, s, slot_c<0>(), slot_c<0>()), load_b(cur, s, slot_c<0>(), slot_c<1>());
                    load_b(cur, s, slot_c<0>(), slot_c<2>()), load_b(cur, s, slot_c<0>(), slot_c<3>());
                    __syncthreads();
                    read_frags(slot_c<0>(), slot_c<0>(), slot_c<0>());
                    read_frags(slot_c<0>(), slot_c<1>(), slot_c<1>());
                    multiply(slot_c<0>(), slot_c<0>());
                    read_frags(slot_c<0>(), slot_c<2>(), slot_c<0>());
                    multiply(slot_c<0>(), slot_c<1>());
                    read_frags(slot_c<0>(), slot_c<3>(), slot_c<1>());
                    multiply(slot_c<0>(), slot_c<2>());
                    multiply(slot_c<0>(), slot_c<3>());
                    if constexpr (kChunked) { // the same two-level accumulation as the pipelined loop
                        if (--until_fold == 0) {
                            total.fold(acc);
                            until_fold = g.chunk_stages;
                        }
                    }
                }
            }
        }

        // Epilogue. Accumulator register v of lane l holds C[8*(v/4) + 4*(l/32) + v%4][l%32] of its 32x32 tile.
        uint32_t const half = lane >> 5, col_in_tile = lane & 31;
        if (T::kUnsigned || NORMS) {
            __syncthreads();
            if constexpr (SELF) {
                if (tid < BM) {
                    if (T::kUnsigned) row_terms[tid] = self_term;
                    if (NORMS) {
                        row_norms[tid] = __builtin_bit_cast(uint32_t, norm_as_f32<T>(self_norm));
                        row_factors[tid] = refined_rsqrt(norm_as_f32<T>(self_norm));
                    }
                }
            }
            // The 8 threads that staged a row left its partial sums in 8 adjacent slots.
            else if (tid < BM) {
                if (T::kUnsigned) {
                    uint32_t const *parts = &row_part[sums_here + tid * 8];
                    uint32_t sum = 0;
#pragma unroll
                    for (int part = 0; part < 8; ++part) sum += parts[part];
                    row_terms[tid] = sum * 128u;
                }
                if (NORMS) {
                    norm_t const *parts = &norm_part[sums_here + tid * 8];
                    norm_t sum = 0;
#pragma unroll
                    for (int part = 0; part < 8; ++part) sum += parts[part];
                    uint32_t bits;
                    if constexpr (sizeof(norm_t) == 8) bits = __builtin_bit_cast(uint32_t, (float)sum); // f64 -> f32, once
                    else bits = (uint32_t)sum;
                    row_norms[tid] = __builtin_bit_cast(uint32_t, norm_as_f32<T>(bits));
                    row_factors[tid] = refined_rsqrt(norm_as_f32<T>(bits));
                }
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < (SELF ? 0 : kLoads); ++i) { // own slots: ready for the tile after next
                if (T::kUnsigned) row_part[sums_here + i * NT + tid] = 0;
                if (NORMS) norm_part[sums_here + i * NT + tid] = 0;
            }
            sums_here ^= (uint32_t)(kLoads * NT);
        }
        // Stores: a scalar base plus one 32-bit per-lane offset, through an explicitly global pointer. (A store
        // through a generic pointer counts as an LDS operation as well, and with such stores in flight the loads
        // prefetched for the next tile could only be waited for all at once.) Tiles that touch the matrix edge take
        // the masked copy of the loop.
        // Of a triangular grid, a wavefront's part of a tile is stored whole (all of it right of the diagonal), not
        // at all (all of it left), or through the masked copy.
        // What only the stores need is read from the kernel's arguments again, here, rather than held in a dozen
        // scalar registers through the loop (the empty asm hides from the compiler that it is the same memory).
        typedef __attribute__((address_space(4))) GemmArgs const late_args_t;
        late_args_t *late = (late_args_t *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(late));
        // Stores go past the caches (`nt`): the output is written once and not read here, and the caches are left to the
        // operands (measured on one box, same run: bf16 8192^3 1.047 -> 0.972 ms, e4m3 1.027 -> 0.933 ms, i8 0.526 ->
        // 0.518 ms, i8 1024 x 1,048,576 x 768 1.455 -> 1.395 ms). Except where the rows of C do not start on 128-byte
        // lines and the product is not deep: a 128-byte run of a row then straddles two lines and would reach the
        // memory as two partial writes; through the L2 the parts of a line written by neighbouring wavefronts meet
        // first (measured, i8, nt -> plain: 8192 x 8191 x 1000
        // 0.199 -> 0.146 ms, 4096 x 4095 x 4096 0.099 -> 0.077, 1024 x 1,000,001 x 768 3.99 -> 1.92 ms; bf16 4096 x 4095 x
        // 4096 0.155 -> 0.143, but 8192 x 8191 x 8192 0.97 -> 1.04: a deep product wants its L2 for the operands).
        // The distance kinds keep `nt` (i8 angular 1024 x 1,000,001 x 768: 2.57 against 2.70 ms).
        bool const lines = (((uint64_t)late->c | late->c_stride) & 127) == 0;
        bool const streamed = NORMS || (late->store_policy ? late->store_policy == 1 : lines || stages > 64);
        // (the distance kinds force the diagonal to zero in the masked copy only: a part of a tile that holds a
        // diagonal element, even its corner alone, is not interior for them)
        bool const interior = row0 + BM <= late->m && col0 + 32 * TN <= late->n &&
                              (((row0 + (BM - 1) + (NORMS ? 1u : 0u) + late->tri_shift) & late->tri_mask) <= col0);
        bool const nothing = ((row0 + late->tri_shift) & late->tri_mask) > col0 + (32 * TN - 1);
        global_u8_t *c_tile = (global_u8_t *)late->c + (uint64_t)row0 * late->c_stride + (uint64_t)col0 * 4;
        auto store_all = [&](auto masked_tag, auto metric_tag, auto streamed_tag) {
            constexpr bool masked = decltype(masked_tag)::value != 0;
            constexpr int metric = decltype(metric_tag)::value;
            constexpr bool past_caches = decltype(streamed_tag)::value != 0;
            uint64_t const row_step = late->c_stride;
            // Lane l holds column l % 32; register v holds row 8 * (v / 4) + 4 * (l / 32) + v % 4.
            uint32_t const lane_offset = 4 * half * (uint32_t)late->c_stride + col_in_tile * 4;
            // Masked tiles: rows of the matrix from this lane's first one on, and how far right of the diagonal
            // col = row + tri_shift its first element lies (element (r, 32 j) from there is stored when
            // r - 32 j <= that distance; without a triangle everything is).
            int const rows_left = (int)(late->m - row0 - 4 * half);
            int const diagonal = late->tri_mask ? (int)(col0 + col_in_tile) - (int)(row0 + 4 * half + late->tri_shift) : 0x7FFFFFFF;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bool const col_ok = col0 + j * 32 + col_in_tile < late->n;
                // Rows come in runs of 4 that start 8 apart: the base advances by one row or by five. The
                // empty asm keeps it a running scalar (otherwise every row's base is precomputed and the
                // scalar registers overflow).
                global_u8_t *row_base = c_tile + j * 128;
                v4i row_term4 = {0, 0, 0, 0}, row_norm4 = {0, 0, 0, 0};
                typedef float v4f __attribute__((ext_vector_type(4)));
                v4f row_factor4 = {0, 0, 0, 0};
                float const col_value = metric != 0 ? norm_as_f32<T>(col_norm[j]) : 0.0f;
                float const col_factor = metric == 1 ? refined_rsqrt(col_value) : 0.0f;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        int const r_fixed = i * 32 + 8 * (v / 4) + (v % 4); // row of lanes 0..31; lanes 32..63 are 4 rows below
                        // a named copy: bit-casting the vector element expression itself reads lane 0
                        auto const element = total.finish(acc, i, j, v);
                        uint32_t bits = finished_dot<T>(__builtin_bit_cast(uint32_t, element));
                        if (T::kUnsigned) {
                            // the terms of 4 consecutive rows in one LDS read
                            if (v % 4 == 0) row_term4 = *(v4i const *)&row_terms[i * 32 + 8 * (v / 4) + 4 * half];
                            bits += (uint32_t)row_term4[v % 4] + col_term[j];
                        }
                        if (metric == 1) {
                            // the cheap form where it is good enough (almost everywhere on vectors that are not near
                            // copies of each other), the full finaliser for the lanes where it is not
                            if (v % 4 == 0) row_factor4 = *(v4f const *)&row_factors[i * 32 + 8 * (v / 4) + 4 * half];
                            bool cheap;
                            float const quick = angular_from_factors<T>(bits, row_factor4[v % 4], col_factor, &cheap);
                            uint32_t result = __builtin_bit_cast(uint32_t, quick);
                            if (__builtin_amdgcn_ballot_w64(!cheap) != 0) { // (uniform: the wavefront branches as one)
                                int const row_bits = *(int const *)&row_norms[i * 32 + 8 * (v / 4) + 4 * half + v % 4];
                                uint32_t const full = distance_from_dot<T, 1>(bits, __builtin_bit_cast(float, row_bits), col_value);
                                result = cheap ? result : full;
                            }
                            bits = result;
                        }
                        else if (metric != 0) {
                            if (v % 4 == 0) row_norm4 = *(v4i const *)&row_norms[i * 32 + 8 * (v / 4) + 4 * half];
                            int const row_bits = row_norm4[v % 4];
                            bits = distance_from_dot<T, 2>(bits, __builtin_bit_cast(float, row_bits), col_value);
                        }
                        bool keep = true;
                        if (masked) {
                            keep = col_ok && r_fixed < rows_left && r_fixed - j * 32 <= diagonal;
                            // a vector's distance from itself is exactly 0 (dots/serial.h:2871-2876)
                            if (metric != 0 && r_fixed - j * 32 == diagonal) bits = 0;
                        }
                        if (keep) {
                            if (past_caches) __builtin_nontemporal_store(bits, (global_u32_t *)(row_base + lane_offset));
                            else *(global_u32_t *)(row_base + lane_offset) = bits;
                        }
                        row_base += (v % 4 == 3 ? 5 : 1) * row_step;
                        asm volatile("" : "+s"(row_base));
                    }
                    // u8 reads a row term per element: keep those reads from being hoisted by the hundred
                    // (registers are what the prefetched tile is short of here).
                    if (T::kUnsigned || metric != 0) __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        auto store_as = [&](auto metric_tag) {
            if (interior) {
                if (NORMS || streamed) store_all(slot_c<0>(), metric_tag, slot_c<1>());
                else if constexpr (!NORMS) store_all(slot_c<0>(), metric_tag, slot_c<0>());
            }
            else {
                if (NORMS || streamed) store_all(slot_c<1>(), metric_tag, slot_c<1>());
                else if constexpr (!NORMS) store_all(slot_c<1>(), metric_tag, slot_c<0>());
            }
        };
        if (nothing) {}
        else if constexpr (NORMS) { // which distance is a run-time choice: one kernel serves both
            if (late->metric == 2) store_as(slot_c<2>());
            else store_as(slot_c<1>());
        }
        else store_as(slot_c<0>());
    }
}

/**
 *  Shallow products, strip by strip. A workgroup of 8 wavefronts keeps the (32*TM) rows of its part of A in LDS, whole depth,
 *  and walks along the columns of C, 256 at a time (a 32-column tile of the image per wavefront). What a tile costs in
 *  dots_packed_kernel besides its own columns (A fetched, masked, widened, its squares and bytes summed, a barrier every
 *  stage) is done once per strip; the loop is B from the image into registers, A fragments from LDS and MFMAs, and the
 *  wavefronts meet only to store.
 *
 *  B is fetched two stages ahead, across tiles, so that what a tile waits for was asked for before the tile before it was
 *  stored (loads and stores of a wavefront complete in order).
 *
 *  Stores are whole 128-byte lines wherever the rows of C start. A partial line costs the memory a read and a write, and
 *  a row's tile ends in the middle of one unless C is aligned to lines: 1000 x 500,009 results written as the accumulators
 *  hold them, 128 bytes per row and instruction, take 1190 us past the caches and 600 through them, as whole lines 400 (the
 *  same as rows on lines). Because a workgroup walks along its rows, what a tile lacks of its first line is what the tile
 *  before it had left over of its last. A row's tile starts `skew` columns past a line; in LDS it starts at the same
 *  position of a row of 256, and its last `skew` columns go around to the row's start. There the first line's missing columns
 *  are filled in from `carried`, and the ones that went around wait there for the next tile.
 */
constexpr int kStripWaves = 8, kStripColumns = 32 * kStripWaves;
template <class T, int TM, int METRIC, int BATCH>
__global__ __launch_bounds__(64 * kStripWaves, 2) void dots_strips_kernel(GemmArgs g) {
    typedef typename T::acc_t acc_t;
    typedef typename T::norm_t norm_t;
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) uint8_t global_u8_t;
    typedef __attribute__((address_space(1))) uint32_t global_u32_t;
    constexpr int BM = TM * 32, NT = 64 * kStripWaves;
    constexpr int kStageLds = BM * kStageBytes;
    constexpr int kSrcStage = kStageChunks * T::kSrcChunk;
    constexpr int kImageTileChunk = kTileRows * T::kImageChunk;
    constexpr bool kChunked = T::kChunked;
    extern __shared__ __attribute__((aligned(1024))) uint8_t strip_lds[];
    uint32_t const stages = g.k_chunks / kStageChunks;
    uint32_t *const stage_rows = (uint32_t *)(strip_lds + stages * kStageLds);    // BATCH rows of 256 results
    uint32_t *const carried = stage_rows + BATCH * kStripColumns;                 // per row what its next line starts with
    uint32_t *const row_terms = carried + BM * 32;                                 // as in dots_packed_kernel
    uint32_t *const row_norms = row_terms + BM;
    float *const row_factors = (float *)(row_norms + BM);

    uint32_t const tid = threadIdx.x, lane = tid & 63;
    uint32_t const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t const half = lane >> 5, col_in_tile = lane & 31;

    PackedHeader const *header = (PackedHeader const *)g.bp;
    bool const image_ok = header->magic == kMagic && header->version == kVersion &&
                          header->dtype == (uint32_t)T::kDtype && header->n == g.n && header->k == g.k &&
                          header->k_chunks == g.k_chunks && header->n_tiles == g.n_tiles;
    uint8_t const *data = g.bp + sizeof(PackedHeader);
    uint32_t const *col_terms = (uint32_t const *)(data + (uint64_t)g.n_tiles * g.k_chunks * kImageTileChunk);
    uint32_t const *col_norms = col_terms + (uint64_t)g.n_tiles * kTileRows;
    uint32_t const strip_columns = g.strip_tiles * kStripColumns;
    if (!image_ok) { // the image was not packed for this call: the reference's error convention, all bits set
        for (uint32_t unit = blockIdx.x; unit < g.tile_count; unit += gridDim.x) {
            uint32_t tile_m, strip;
            tile_of_block(unit, g, tile_m, strip);
            for (uint32_t row = tile_m * BM; row < tile_m * BM + BM && row < g.m; ++row)
                for (uint32_t at = tid; at < strip_columns; at += NT)
                    if (strip * strip_columns + at < g.n) *(global_u32_t *)((global_u8_t *)g.c + (uint64_t)row * g.c_stride + (uint64_t)(strip * strip_columns + at) * 4) = 0xFFFFFFFFu;
        }
        return;
    }

    uint32_t a_frag[4]; // (lane l takes row l % 32 of each 32-row block and chunk 2q + l / 32)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t const r = lane & 31, c = 2 * q + (lane >> 5);
        a_frag[q] = r * kStageBytes + ((c ^ ((r >> 1) & 7)) << 4);
    }
    uint32_t const tile_bytes = g.k_chunks * kImageTileChunk;
    struct ImageView {
        uint8_t const *b;
        uint32_t bytes;
    };
    auto view_of = [&](uint32_t col0) { // (columns past the last tile: that tile once more, never stored)
        uint32_t const tile = col0 / 32 < g.n_tiles ? col0 / 32 : g.n_tiles - 1;
        uint64_t const left = (uint64_t)(g.n_tiles - tile) * tile_bytes;
        return ImageView {data + (uint64_t)tile * tile_bytes, left < 0xFFFFFFFFull ? (uint32_t)left : 0xFFFFFFFFu};
    };
    v4i b_reg[2][4];
    v4i af[2][TM];
    acc_t acc[TM][1];
    Totals<acc_t, TM, 1, kChunked> total;
    auto load_b = [&](ImageView const &view, uint32_t s, auto slot_tag, auto q_tag) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_tag)::value, q = decltype(q_tag)::value;
        __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)view.b, 0, (int)view.bytes, 0x00020000);
        uint32_t const offset = __builtin_amdgcn_readfirstlane(s * (kStageChunks * kImageTileChunk));
        if constexpr (T::kImageChunk == 2)
            b_reg[slot][q][0] = (int)(uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, lane * 2 + q * 2 * kImageTileChunk, offset, 0);
        else
            b_reg[slot][q] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16 + q * 2 * kImageTileChunk, offset, 0));
    };
    auto read_frags = [&](uint32_t stage_at, auto q_tag, auto parity_tag) __attribute__((always_inline)) {
        constexpr int q = decltype(q_tag)::value, parity = decltype(parity_tag)::value;
        uint8_t const *src = strip_lds + stage_at + a_frag[q];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[parity][i] = *(v4i const *)(src + i * 32 * kStageBytes);
    };
    auto multiply = [&](auto slot_tag, auto q_tag, auto entry_tag) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_tag)::value, q = decltype(q_tag)::value, entry = decltype(entry_tag)::value;
        v4i const b = T::operand_b(b_reg[slot][q]);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (entry == 0) T::mma(acc[i][0], af[q & 1][i], b);
            else {
                if constexpr (entry == 1) total.fold_block(acc, i, 0);
                else total.clear_block(i, 0);
                T::mma_fresh(acc[i][0], af[q & 1][i], b);
            }
        }
    };
    auto schedule_k_step = [&](auto vector_tag) __attribute__((always_inline)) {
        constexpr int vector = decltype(vector_tag)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (vector > 0) __builtin_amdgcn_sched_group_barrier(0x002, vector, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto meet = [&]() __attribute__((always_inline)) { // (orders LDS only: prefetched loads and stores stay in flight)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    // Where in the LDS rows a lane's results go, in bytes, two to a register: 16 rows of each 32-row block, the same in all
    // of them (32 rows further on a row's start has moved by whole lines).
    uint32_t places[4][2];
#pragma unroll
    for (int quad = 0; quad < 4; ++quad)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            uint32_t const words = (uint32_t)((uint64_t)g.c >> 2) + (8 * quad + 4 * half + e) * (uint32_t)(g.c_stride >> 2);
            uint32_t const even = ((words & 31) + 32 * wave + col_in_tile) & (kStripColumns - 1);
            uint32_t const odd = (((words + (uint32_t)(g.c_stride >> 2)) & 31) + 32 * wave + col_in_tile) & (kStripColumns - 1);
            places[quad][e / 2] = (even * 4 + half * (4 * 4 * kStripColumns)) | (odd * 4 + half * (4 * 4 * kStripColumns)) << 16;
        }

    for (uint32_t unit = blockIdx.x; unit < g.tile_count; unit += gridDim.x) {
        uint32_t tile_m, strip;
        tile_of_block(unit, g, tile_m, strip);
        uint32_t const row0 = tile_m * BM, strip_col = strip * strip_columns;
        if (strip_col >= g.n) continue;
        // The part of A. Thread t takes chunk t % 8 of every stage of rows t / 8, t / 8 + 64, ...: the partial sums of a row
        // are those of dots_packed_kernel, in the same order.
        meet(); // (the strip before is done with the LDS)
        {
            uint32_t *const part_sums = stage_rows;       // (BM x 8 of them)
            norm_t *const part_norms = (norm_t *)carried; // (and as many of these)
            static_assert(BM * 8 <= BATCH * kStripColumns && BM * 8 * sizeof(norm_t) <= BM * 32 * sizeof(uint32_t), "partial sums: they fit where they wait");
            uint32_t const a_pos = tid & 7;
            for (uint32_t r = tid >> 3; r < (uint32_t)BM; r += NT / 8) {
                bool const exists = row0 + r < g.m;
                uint8_t const *source = g.a + (uint64_t)(exists ? row0 + r : g.m - 1) * g.a_stride + a_pos * T::kSrcChunk;
                uint32_t sum = 0;
                norm_t squares = 0;
#pragma unroll 4
                for (uint32_t s = 0; s < stages; ++s) {
                    int64_t const left = (int64_t)g.k_src_bytes - (int64_t)s * kSrcStage - (int64_t)a_pos * T::kSrcChunk;
                    int const valid = (int)(left > T::kSrcChunk ? T::kSrcChunk : (left < 0 ? 0 : left));
                    v4i v = load_chunk_guarded<T::kSrcChunk>(source + (uint64_t)s * kSrcStage, valid, 0u);
                    v4i const raw = v;
                    if (T::kUnsigned) {
                        sum += sum_bytes_u8(v);
#pragma unroll
                        for (int w = 0; w < 4; ++w) { // flip only bytes that exist: the zero padding stays zero
                            int const rem = valid - 4 * w;
                            v[w] ^= (int)(rem >= 4 ? 0x80808080u : (rem <= 0 ? 0u : (0x80808080u >> (8 * (4 - rem)))));
                        }
                    }
                    v4i const wide = T::widen(v);
                    if (METRIC != 0) squares += T::sumsq(raw, wide);
                    *(v4i *)(strip_lds + s * kStageLds + r * kStageBytes + ((a_pos ^ ((r >> 1) & 7)) << 4)) = wide;
                }
                if (T::kUnsigned) part_sums[r * 8 + a_pos] = sum;
                if (METRIC != 0) part_norms[r * 8 + a_pos] = squares;
            }
            meet();
            if ((T::kUnsigned || METRIC != 0) && tid < BM) {
                if (T::kUnsigned) {
                    uint32_t sum = 0;
#pragma unroll
                    for (int part = 0; part < 8; ++part) sum += part_sums[tid * 8 + part];
                    row_terms[tid] = sum * 128u;
                }
                if (METRIC != 0) {
                    norm_t sum = 0;
#pragma unroll
                    for (int part = 0; part < 8; ++part) sum += part_norms[tid * 8 + part];
                    uint32_t bits;
                    if constexpr (sizeof(norm_t) == 8) bits = __builtin_bit_cast(uint32_t, (float)sum);
                    else bits = (uint32_t)sum;
                    row_norms[tid] = __builtin_bit_cast(uint32_t, norm_as_f32<T>(bits));
                    row_factors[tid] = refined_rsqrt(norm_as_f32<T>(bits));
                }
            }
            meet();
        }

        ImageView cur = view_of(strip_col + 32 * wave);
        auto load_stage = [&](auto slot_tag) __attribute__((always_inline)) {
            constexpr int slot = decltype(slot_tag)::value;
            load_b(cur, slot, slot_tag, slot_c<0>()), load_b(cur, slot, slot_tag, slot_c<1>());
            load_b(cur, slot, slot_tag, slot_c<2>()), load_b(cur, slot, slot_tag, slot_c<3>());
        };
        load_stage(slot_c<0>()), load_stage(slot_c<1>());
        auto column_at = [&](uint32_t col0) { return (col0 / 32 < g.n_tiles ? col0 / 32 : g.n_tiles - 1) * kTileRows + col_in_tile; };
        uint32_t col_term = 0, col_norm = 0;
        if (T::kUnsigned) col_term = col_terms[column_at(strip_col + 32 * wave)];
        if (METRIC != 0) col_norm = col_norms[column_at(strip_col + 32 * wave)];
        read_frags(0, slot_c<0>(), slot_c<0>());

        for (uint32_t tile = 0; tile < g.strip_tiles; ++tile) {
            uint32_t const tile_col = strip_col + tile * kStripColumns;
            if (tile_col >= g.n + 32) break; // (nothing left, not even of a last line; uniform)
            uint32_t const next_col = tile_col + kStripColumns + 32 * wave;
            ImageView const nxt = view_of(next_col);
            auto stage = [&](auto slot_tag, uint32_t s, auto entry_tag) __attribute__((always_inline)) {
                constexpr int entry = decltype(entry_tag)::value;
                bool const wrap = s + 2 >= stages;
                uint32_t const ahead = wrap ? s + 2 - stages : s + 2;
                ImageView const &from = wrap ? nxt : cur;
                uint32_t const here = s * kStageLds, after = s + 1 < stages ? here + kStageLds : 0;
                __builtin_amdgcn_sched_barrier(0);
                read_frags(here, slot_c<1>(), slot_c<1>());
                multiply(slot_tag, slot_c<0>(), entry_tag);
                load_b(from, ahead, slot_tag, slot_c<0>());
                schedule_k_step(slot_c<kChunked && entry != 0 ? 16 : 0>());
                read_frags(here, slot_c<2>(), slot_c<0>());
                multiply(slot_tag, slot_c<1>(), slot_c<0>());
                load_b(from, ahead, slot_tag, slot_c<1>());
                schedule_k_step(slot_c<0>());
                read_frags(here, slot_c<3>(), slot_c<1>());
                multiply(slot_tag, slot_c<2>(), slot_c<0>());
                load_b(from, ahead, slot_tag, slot_c<2>());
                schedule_k_step(slot_c<0>());
                read_frags(after, slot_c<0>(), slot_c<0>());
                multiply(slot_tag, slot_c<3>(), slot_c<0>());
                load_b(from, ahead, slot_tag, slot_c<3>());
                schedule_k_step(slot_c<0>());
            };
            stage(slot_c<0>(), 0u, slot_c<2>());
            stage(slot_c<1>(), 1u, slot_c<0>());
            for (uint32_t s = 2; s < stages; s += 2) { // (two-accumulator types: the sums go into the totals every two stages)
                stage(slot_c<0>(), s, slot_c<kChunked ? 1 : 0>());
                stage(slot_c<1>(), s + 1, slot_c<0>());
            }
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
            uint32_t const my_term = col_term, my_norm = col_norm;
            if (T::kUnsigned) col_term = col_terms[column_at(next_col)]; // (asked for in front of the stores)
            if (METRIC != 0) col_norm = col_norms[column_at(next_col)];

            // Buffer stores: rows past the last one lie behind the descriptor's end, and so does the offset of a column that is
            // not to be stored. (All of the offset is the lane's: the range check takes a scalar offset off the
            // descriptor's size, which rows past the end would make negative.)
            typedef __attribute__((address_space(4))) GemmArgs const late_args_t;
            late_args_t *late = (late_args_t *)__builtin_amdgcn_kernarg_segment_ptr();
            asm volatile("" : "+s"(late));
            constexpr int kRowLanes = NT / BATCH; // threads that store a row
            float const col_value = METRIC != 0 ? norm_as_f32<T>(my_norm) : 0.0f;
            float const col_factor = METRIC == 1 ? refined_rsqrt(col_value) : 0.0f;
            uint32_t const row_step = (uint32_t)late->c_stride, n = late->n;
            uint32_t const words = (uint32_t)((uint64_t)late->c >> 2), step = row_step >> 2;
            constexpr uint32_t kNowhere = 0x80000000u; // (the host checks that a tile's rows end below it)
            uint8_t *const c_tile = late->c + (uint64_t)row0 * late->c_stride + (uint64_t)tile_col * 4 - 128;
            uint64_t const left = (uint64_t)(late->m - row0 - 1) * late->c_stride + (uint64_t)n * 4 - (uint64_t)tile_col * 4 + 128;
            __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)c_tile, 0, (int)(left < kNowhere ? (uint32_t)left : kNowhere), 0x00020000);
            bool const inner = tile != 0 && tile_col + kStripColumns <= n;
            bool const last = tile + 1 == g.strip_tiles;
#pragma unroll
            for (int batch = 0; batch < BM / BATCH; ++batch) {
                int const i = batch * BATCH / 32;
#pragma unroll
                for (int quad = 0; quad < BATCH / 8; ++quad) {
                    int const row_quad = (batch * BATCH % 32) / 8 + quad; // run of four rows per lane, of the 32 of block i
                    int const rows_at = i * 32 + 8 * row_quad + 4 * half;
                    v4i row_term4 = {0, 0, 0, 0}, row_norm4 = {0, 0, 0, 0};
                    v4f row_factor4 = {0, 0, 0, 0};
                    if (T::kUnsigned) row_term4 = *(v4i const *)&row_terms[rows_at];
                    if (METRIC == 1) row_factor4 = *(v4f const *)&row_factors[rows_at];
                    if (METRIC == 2) row_norm4 = *(v4i const *)&row_norms[rows_at];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        auto const element = total.finish(acc, i, 0, 4 * row_quad + e);
                        uint32_t bits = finished_dot<T>(__builtin_bit_cast(uint32_t, element));
                        if (T::kUnsigned) bits += (uint32_t)row_term4[e] + my_term;
                        if (METRIC == 1) {
                            bool cheap;
                            float const quick = angular_from_factors<T>(bits, row_factor4[e], col_factor, &cheap);
                            uint32_t result = __builtin_bit_cast(uint32_t, quick);
                            if (__builtin_amdgcn_ballot_w64(!cheap) != 0) {
                                int const row_bits = *(int const *)&row_norms[rows_at + e];
                                uint32_t const full = distance_from_dot<T, 1>(bits, __builtin_bit_cast(float, row_bits), col_value);
                                result = cheap ? result : full;
                            }
                            bits = result;
                        }
                        else if (METRIC == 2) {
                            int const row_bits = row_norm4[e];
                            bits = distance_from_dot<T, 2>(bits, __builtin_bit_cast(float, row_bits), col_value);
                        }
                        uint32_t const pair = places[row_quad][e / 2], place = e % 2 ? pair >> 16 : pair & 0xFFFFu;
                        *(uint32_t *)((uint8_t *)(stage_rows + (8 * quad + e) * kStripColumns) + place) = bits;
                    }
                }
                meet();
                uint32_t const row_in_batch = tid / kRowLanes, row = batch * BATCH + row_in_batch;
                uint32_t const skew = (words + row * step) & 31;
                uint32_t const row_at = row * row_step;
#pragma unroll
                for (int part = 0; part < kStripColumns / 4 / kRowLanes; ++part) {
                    uint32_t const chunk = part * kRowLanes + tid % kRowLanes; // sixteen bytes of the row's lines
                    v4u const fresh = *(v4u const *)&stage_rows[row_in_batch * kStripColumns + 4 * chunk];
                    v4u values = fresh;
                    uint32_t const target = row_at + (32 - skew + 4 * chunk) * 4;
                    int const column = (int)(tile_col - skew + 4 * chunk);
                    if (part == 0 && chunk < 8) {
                        v4u *const waiting = (v4u *)&carried[row * 32 + 4 * chunk];
                        v4u const before = *waiting;
                        *waiting = fresh;
#pragma unroll
                        for (int e = 0; e < 4; ++e) values[e] = 4 * chunk + e < skew ? before[e] : fresh[e];
                        if (last) { // the end of the strip: what the last line of every row still lacks
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                bool const mine = 4 * chunk + e < skew && column + kStripColumns + e < (int)n;
                                __builtin_amdgcn_raw_buffer_store_b32(fresh[e], rsrc, mine ? target + 4 * kStripColumns + 4 * e : kNowhere, 0, 0);
                            }
                        }
                    }
                    if (inner) __builtin_amdgcn_raw_buffer_store_b128(values, rsrc, target, 0, 2); // (2: `nt`)
                    else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            bool const mine = column + e >= (int)strip_col && column + e < (int)n;
                            __builtin_amdgcn_raw_buffer_store_b32(values[e], rsrc, mine ? target + 4 * e : kNowhere, 0, 0);
                        }
                    }
                }
                meet();
            }
        }
    }
}

/**
 *  Shallow products into a large C with A in registers. A workgroup of 8 wavefronts holds its rows of A (32*TM per wavefront, whole
 *  depth) as the MFMA wants them and walks along the columns of C, one 32-column tile of the image at a time. The tile comes straight
 *  from the image, which lies in the order of the fragments, into a ring of LDS tiles, kSlots - 1 ahead; every wavefront reads it there,
 *  multiplies it with its own rows and stores 128 bytes of each. One barrier per tile, and nothing is staged.
 *
 *  Why: such products are bound by the memory, and what keeps a copy's rate from them is the reading. Writes of C in any of the shapes
 *  below reach 4.9 TB/s, and reads of as many bytes as B has beside them take their own time more (1024 x 1,048,576 results and 768 bytes a
 *  column, no arithmetic: 872 us written, 130 read, 1030 to 1040 both, as long as every byte is asked for once), but with every line of B
 *  asked for by eight workgroups at about the same time, as tiles of 128 rows do, both take 1280, however far ahead they ask: what a
 *  compute unit reads waits in one queue with what it writes. Here B is read once per 256 rows (TM 1) or 512.
 *
 *  Whole calls, before and now (us): i8 1024 x 1,048,576 x 768 1363 (256 x 256 tiles) and 1080, 1000 x 500,032 x 700 803 and 557, f16
 *  8192 x 8191 x 500 149 (strips) and 104, 1000 x 300,009 x 600 650 and 481, i8 angular 1024 x 524,288 x 768 870 and 667; the same bits.
 *
 *  CARRY: rows of C that do not start on 128-byte lines. What is stored is whole lines all the same: the results of a row are
 *  rotated by its distance from a line (ds_bpermute), and what belongs to its next line waits in registers for the next tile.
 */
constexpr int kResidentWaves = 8;
template <class T, int TM, int STAGES, int METRIC, bool CARRY>
__global__ __launch_bounds__(64 * kResidentWaves, 2) void dots_resident_kernel(GemmArgs g) {
    typedef typename T::acc_t acc_t;
    typedef typename T::norm_t norm_t;
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) uint8_t global_u8_t;
    typedef __attribute__((address_space(1))) uint32_t global_u32_t;
    constexpr int BM = TM * 32, kSteps = STAGES * 4, kRows = kResidentWaves * BM;
    constexpr int kStepBytes = 1024; // of a 32-column tile, what one MFMA step takes
    static_assert(T::kImageChunk == 16, "the image holds the fragments");
    constexpr int kTileBytes = kSteps * kStepBytes;
    constexpr int kSlots = STAGES > 8 ? 3 : 4;
    constexpr int kFetches = kTileBytes / 1024 / kResidentWaves; // per wavefront and tile
    static_assert(kFetches * kResidentWaves * 1024 == kTileBytes, "every wavefront fetches as much: the waits count on it");
    constexpr bool kChunked = T::kChunked;
    // (three kernels whose registers fit only with two fragments read ahead: with three they reloaded 8 (u8, e2m3) and 16 (u4) of them in
    // front of every tile's MFMAs, behind the stores. Means over 444 to 513 shapes each, against the tiles or strips they replace: u8 0.93
    // and 0.82 of the time, u4 1.01 and 0.79, e2m3 0.93 and 0.82)
    constexpr bool kTight = CARRY && STAGES == 10 && METRIC == 1 && (T::kDtype == kU8 || T::kDtype == kU4 || T::kDtype == kE2M3);
    __shared__ __attribute__((aligned(1024))) uint8_t ring0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t ring1[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t ring2[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t ring3[kSlots > 3 ? kTileBytes : 16];
    __shared__ __attribute__((aligned(16))) uint32_t row_terms[T::kUnsigned ? kRows : 4]; // as in dots_packed_kernel
    __shared__ __attribute__((aligned(16))) uint32_t row_norms[METRIC != 0 ? kRows : 4];
    __shared__ __attribute__((aligned(16))) float row_factors[METRIC == 1 ? kRows : 4];
    uint32_t const tid = threadIdx.x, lane = tid & 63;
    uint32_t const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t const half = lane >> 5, col_in_tile = lane & 31;

    PackedHeader const *header = (PackedHeader const *)g.bp;
    bool const image_ok = header->magic == kMagic && header->version == kVersion &&
                          header->dtype == (uint32_t)T::kDtype && header->n == g.n && header->k == g.k &&
                          header->k_chunks == g.k_chunks && header->n_tiles == g.n_tiles;
    uint8_t const *data = g.bp + sizeof(PackedHeader);
    uint32_t const *col_terms = (uint32_t const *)(data + (uint64_t)g.n_tiles * kTileBytes);
    uint32_t const *col_norms = col_terms + (uint64_t)g.n_tiles * kTileRows;
    uint32_t const waves = g.strip_waves, block_rows = waves * BM; // (the wavefronts that have rows)
    uint32_t tile_m, strip;
    tile_of_block(blockIdx.x, g, tile_m, strip);
    uint32_t const first = strip * g.strip_tiles;
    if (first >= g.n_tiles) return;
    uint32_t const count = g.n_tiles - first < g.strip_tiles ? g.n_tiles - first : g.strip_tiles;
    if (!image_ok) { // the image was not packed for this call: the reference's error convention, all bits set
        for (uint32_t row = tile_m * block_rows; row < tile_m * block_rows + block_rows && row < g.m; ++row)
            for (uint32_t col = first * 32 + tid; col < (first + count) * 32 && col < g.n; col += 64 * kResidentWaves)
                *(global_u32_t *)((global_u8_t *)g.c + (uint64_t)row * g.c_stride + (uint64_t)col * 4) = 0xFFFFFFFFu;
        return;
    }
    uint32_t const row0 = tile_m * block_rows + wave * BM;
    bool const works = wave < waves && row0 < g.m; // (a wavefront without rows helps to fetch)

    auto ring_of = [&](auto slot_tag) -> uint8_t * {
        constexpr int slot = decltype(slot_tag)::value % kSlots;
        return slot == 0 ? ring0 : (slot == 1 ? ring1 : (slot == 2 ? ring2 : ring3));
    };
    // Tile t of the strip on its way into LDS, 1 KiB per instruction (past the strip's end its last one again, which nobody reads).
    auto fetch = [&](uint32_t t, auto slot_tag) __attribute__((always_inline)) {
        uint32_t const tile = __builtin_amdgcn_readfirstlane(first + (t < count ? t : count - 1));
        __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(data + (uint64_t)tile * kTileBytes), 0, kTileBytes, 0x00020000);
#pragma unroll
        for (int at = 0; at < kFetches * kResidentWaves; at += kResidentWaves)
            fetch_to_lds(rsrc, (lds_void_t *)(ring_of(slot_tag) + (at + wave) * 1024), (at + wave) * 1024 + lane * 16, 0);
    };
    fetch(0, slot_c<0>()), fetch(1, slot_c<1>());
    if constexpr (kSlots > 3) fetch(2, slot_c<2>());

    // The wavefront's rows of A: lane l takes row l % 32 of each 32-row block and chunk 2q + l / 32. Rows may start on any byte:
    // the aligned dwords that hold a chunk, one more than the chunk has, and a shift.
    v4i a[kSteps][TM];
    if (works) {
        uint32_t const skew = (uint32_t)((uint64_t)g.a + (uint64_t)row0 * g.a_stride) & 3u;
        uint8_t const *base = g.a + (uint64_t)row0 * g.a_stride - skew;
        uint32_t const rows_here = g.m - row0 < (uint32_t)BM ? g.m - row0 : (uint32_t)BM;
        uint32_t const bytes = (skew + (rows_here - 1) * (uint32_t)g.a_stride + (uint32_t)g.k_src_bytes + 3u) & ~3u;
        __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, 0x00020000);
        constexpr int kWords = (T::kSrcChunk + 3) / 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            uint32_t const at = skew + (i * 32 + col_in_tile) * (uint32_t)g.a_stride + half * T::kSrcChunk, shift = at & 3u;
            uint32_t sum = 0;
            norm_t squares[4] = {0, 0, 0, 0}; // (of the chunks at positions 2 * (q % 4) + half of their stages)
#pragma unroll
            for (int q = 0; q < kSteps; ++q) {
                uint32_t const offset = (at & ~3u) + 2 * q * T::kSrcChunk;
                uint32_t word[5] = {0, 0, 0, 0, 0};
                if constexpr (T::kSrcChunk == 16) {
                    v4i const wide = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0));
                    word[0] = (uint32_t)wide[0], word[1] = (uint32_t)wide[1], word[2] = (uint32_t)wide[2], word[3] = (uint32_t)wide[3];
                    word[4] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, offset + 16, 0, 0);
                }
                else {
                    typedef unsigned v3u __attribute__((ext_vector_type(3)));
                    v3u const narrow = __builtin_amdgcn_raw_buffer_load_b96(rsrc, offset, 0, 0);
                    word[0] = narrow[0], word[1] = narrow[1], word[2] = narrow[2];
                }
                v4i v = {0, 0, 0, 0};
#pragma unroll
                for (int w = 0; w < kWords; ++w) v[w] = (int)__builtin_amdgcn_alignbyte(word[w + 1], word[w], shift);
                // (the depth ends in the last two stages: what lies behind a row's end is cleared where the arithmetic cares)
                uint32_t exists[kWords];
#pragma unroll
                for (int w = 0; w < kWords; ++w) {
                    exists[w] = 0xFFFFFFFFu;
                    if (tail_matters_for<T, METRIC != 0>() && q >= kSteps - 8) {
                        int const over = (int)(uint32_t)g.k_src_bytes - (int)((2 * q + half) * T::kSrcChunk) - 4 * w, left = over < 0 ? 0 : (over > 4 ? 4 : over);
                        exists[w] = left == 4 ? 0xFFFFFFFFu : ((1u << (8 * left)) - 1u);
                        v[w] &= (int)exists[w];
                    }
                }
                v4i const raw = v;
                if constexpr (T::kUnsigned) {
                    sum += sum_bytes_u8(v);
#pragma unroll
                    for (int w = 0; w < kWords; ++w) v[w] ^= (int)(exists[w] & 0x80808080u); // (the zeros behind a row's end stay zeros)
                }
                v4i const wide = T::widen(v);
                if constexpr (METRIC != 0) squares[q % 4] += T::sumsq(raw, wide);
                a[q][i] = wide;
                if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            uint32_t const other = (lane ^ 32) * 4, row = wave * BM + i * 32 + col_in_tile;
            if constexpr (T::kUnsigned) {
                sum += (uint32_t)__builtin_amdgcn_ds_bpermute((int)other, (int)sum);
                if (!half) row_terms[row] = sum * 128u;
            }
            if constexpr (METRIC != 0) {
                norm_t total = 0;
#pragma unroll
                for (int position = 0; position < 8; ++position) { // (the order of dots_packed_kernel)
                    norm_t theirs;
                    norm_t const mine = squares[position / 2];
                    if constexpr (sizeof(norm_t) == 8) {
                        uint64_t const bits = __builtin_bit_cast(uint64_t, mine);
                        uint64_t const low = (uint32_t)__builtin_amdgcn_ds_bpermute((int)other, (int)(uint32_t)bits);
                        uint64_t const high = (uint32_t)__builtin_amdgcn_ds_bpermute((int)other, (int)(uint32_t)(bits >> 32));
                        theirs = __builtin_bit_cast(norm_t, low | high << 32);
                    }
                    else theirs = (norm_t)__builtin_amdgcn_ds_bpermute((int)other, (int)mine);
                    total += (position & 1) == (int)half ? mine : theirs;
                }
                uint32_t bits;
                if constexpr (sizeof(norm_t) == 8) bits = __builtin_bit_cast(uint32_t, (float)total);
                else bits = (uint32_t)total;
                if (!half) {
                    row_norms[row] = __builtin_bit_cast(uint32_t, norm_as_f32<T>(bits));
                    if (METRIC == 1) row_factors[row] = refined_rsqrt(norm_as_f32<T>(bits));
                }
            }
        }
    }
    auto column_of = [&](uint32_t t) { return (first + (t < count ? t : count - 1)) * kTileRows + col_in_tile; };
    uint32_t col_term = 0, col_norm = 0;
    if (T::kUnsigned) col_term = col_terms[column_of(0)];
    if (METRIC != 0) col_norm = col_norms[column_of(0)];

    acc_t acc[TM], total[kChunked ? TM : 1];
    // Own fetches of the tile first (all but the `later` youngest vector memory operations have to be done), then everybody's. No
    // fence: that would wait for the later tiles as well.
    auto arrived = [&](auto later_tag) __attribute__((always_inline)) {
        constexpr int later = decltype(later_tag)::value;
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | (later & 15) | (later >> 4) << 14); // (and this wavefront's LDS reads are done)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t carried[CARRY ? TM : 1][CARRY ? 16 : 1];
    uint32_t const step4 = CARRY ? (uint32_t)g.c_stride & 127u : 0u; // how much further from a line the next row starts, in bytes
    uint32_t const skew4 = CARRY ? ((uint32_t)(uint64_t)g.c + (row0 + 4 * half) * (uint32_t)g.c_stride) & 127u : 0u;
    // A tile issues TM * 16 stores at least whatever of it exists (what does not is stored nowhere: past the end of the descriptor), so
    // that this many operations at least are younger than its fetches when a tile is waited for.
    constexpr int kLater = (kSlots - 1) * TM * 16 + (kSlots - 2) * kFetches;
    auto tile = [&](uint32_t t, auto slot_tag) __attribute__((always_inline)) {
        arrived(slot_c<(kLater < 62 ? kLater : 62)>());
        fetch(t + kSlots - 1, slot_c<decltype(slot_tag)::value + kSlots - 1>());
        uint8_t const *src = ring_of(slot_tag) + lane * 16;
        constexpr int kAhead = (TM == 2 && STAGES == 6) || kTight ? 2 : 3; // (fragments read ahead: registers are short there)
        v4i b[4];
        auto read_b = [&](int q) __attribute__((always_inline)) {
            b[q & 3] = *(v4i const *)(src + q * kStepBytes);
        };
        read_b(0), read_b(1);
        if constexpr (kAhead > 2) read_b(2);
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            if (q + kAhead < kSteps) read_b(q + kAhead);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (kChunked && q % 8 == 0) { // (two-accumulator types: the sums go into the totals every two stages)
                    if (q == 0) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) total[i][v] = 0;
                    }
                    else total[i] += acc[i];
                }
                if (q == 0 || (kChunked && q % 8 == 0)) T::mma_fresh(acc[i], a[q][i], b[q & 3]);
                else T::mma(acc[i], a[q][i], b[q & 3]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        uint32_t const my_term = col_term, my_norm = col_norm;
        if (T::kUnsigned) col_term = col_terms[column_of(t + 1)]; // (asked for in front of the stores)
        if (METRIC != 0) col_norm = col_norms[column_of(t + 1)];
        uint32_t const col0 = (first + t) * 32;
        typedef __attribute__((address_space(4))) GemmArgs const late_args_t;
        late_args_t *late = (late_args_t *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(late));
        constexpr uint32_t kNowhere = 0x80000000u; // (the host checks that a wavefront's rows end below it)
        uint32_t const row_step = (uint32_t)late->c_stride, n = late->n;
        // (CARRY: from a line further left, so that offsets of lines that start in front of the tile are not negative)
        uint8_t *const c_tile = late->c + (uint64_t)row0 * late->c_stride + (uint64_t)col0 * 4 - (CARRY ? 128 : 0);
        uint64_t const left = (uint64_t)(late->m - row0 - 1) * late->c_stride + ((uint64_t)n - col0) * 4 + (CARRY ? 128 : 0);
        __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)c_tile, 0, (int)(left < kNowhere ? (uint32_t)left : kNowhere), 0x00020000);
        int const cols_left = (int)(n - col0); // of columns from this tile's first on
        float const col_value = METRIC != 0 ? norm_as_f32<T>(my_norm) : 0.0f;
        float const col_factor = METRIC == 1 ? refined_rsqrt(col_value) : 0.0f;
        // (Results finished before any is stored. u8 euclidean of twelve stages: 25 registers were reloaded with every tile with 16 of them;
        // 599 shapes 0.97 and 0.75 of the time of what it replaces)
        constexpr int kGroup = CARRY || (T::kDtype == kU8 && STAGES == 12 && METRIC == 2) ? 8 : 16;
        auto store_all = [&](auto edge_tag) __attribute__((always_inline)) {
            constexpr bool edge = decltype(edge_tag)::value != 0; // (CARRY) the strip's first tile or its last
            uint32_t offset = 4 * half * row_step + col_in_tile * 4;
            if (CARRY) offset += 128;
            else offset = (int)col_in_tile < cols_left ? offset : kNowhere;
            // (the empty asm keeps these two from being worked out for every row once and held in registers)
            uint32_t moved = skew4, lane4 = col_in_tile * 4;
            if (CARRY) asm volatile("" : "+v"(moved), "+v"(lane4));
            uint32_t moved_again = moved;
            v4i row_term4 = {0, 0, 0, 0}, row_norm4 = {0, 0, 0, 0};
            v4f row_factor4 = {0, 0, 0, 0};
#pragma unroll
            for (int group = 0; group < TM * 16 / kGroup; ++group) {
                int const i = group * kGroup / 16, v0 = group * kGroup % 16;
                uint32_t finished[kGroup];
#pragma unroll
                for (int v = v0; v < v0 + kGroup; ++v) {
                    uint32_t const rows_at = wave * BM + i * 32 + 8 * (v / 4) + 4 * half;
                    auto element = acc[i][v];
                    if constexpr (kChunked) element += total[i][v];
                    uint32_t bits = finished_dot<T>(__builtin_bit_cast(uint32_t, element));
                    if (T::kUnsigned) {
                        if (v % 4 == 0) row_term4 = *(v4i const *)&row_terms[rows_at];
                        bits += (uint32_t)row_term4[v % 4] + my_term;
                    }
                    if (METRIC == 1) {
                        if (v % 4 == 0) row_factor4 = *(v4f const *)&row_factors[rows_at];
                        bool cheap;
                        float const quick = angular_from_factors<T>(bits, row_factor4[v % 4], col_factor, &cheap);
                        uint32_t result = __builtin_bit_cast(uint32_t, quick);
                        if (__builtin_amdgcn_ballot_w64(!cheap) != 0) {
                            int const row_bits = *(int const *)&row_norms[rows_at + v % 4];
                            uint32_t const full = distance_from_dot<T, 1>(bits, __builtin_bit_cast(float, row_bits), col_value);
                            result = cheap ? result : full;
                        }
                        bits = result;
                    }
                    else if (METRIC == 2) {
                        if (v % 4 == 0) row_norm4 = *(v4i const *)&row_norms[rows_at];
                        int const row_bits = row_norm4[v % 4];
                        bits = distance_from_dot<T, 2>(bits, __builtin_bit_cast(float, row_bits), col_value);
                    }
                    finished[v - v0] = bits;
                    if constexpr (CARRY) { // Lane p of a row that starts `moved` bytes past a line takes column p - moved / 4 of the tile.
                        uint32_t const from = (lane4 - moved) & 124u;
                        finished[v - v0] = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(from | half * 128), (int)bits);
                        moved = (moved + (v % 4 == 3 ? 5 : 1) * step4) & 127u;
                    }
                    if ((T::kUnsigned || METRIC != 0) && v % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int v = v0; v < v0 + kGroup; ++v) {
                    uint32_t bits = finished[v - v0], at = offset;
                    if constexpr (CARRY) { // What belongs to the row's line before, this tile's first lanes, was left by the tile before.
                        bool const before = lane4 < moved_again;
                        bits = before ? carried[i][v] : finished[v - v0];
                        carried[i][v] = finished[v - v0];
                        at = offset - moved_again;
                        if (edge) {
                            int const column4 = (int)(lane4 - moved_again);
                            if (t + 1 == count) // the end of the strip: what the last line of every row still lacks
                                __builtin_amdgcn_raw_buffer_store_b32(finished[v - v0], rsrc, before && column4 + 128 < 4 * cols_left ? at + 128 : kNowhere, 0, 2);
                            at = (t != 0 || !before) && column4 < 4 * cols_left ? at : kNowhere;
                        }
                        moved_again = (moved_again + (v % 4 == 3 ? 5 : 1) * step4) & 127u;
                    }
                    __builtin_amdgcn_raw_buffer_store_b32(bits, rsrc, at, 0, 2); // (2: `nt`)
                    offset += (v % 4 == 3 ? 5 : 1) * row_step;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (!CARRY || (t != 0 && t + 1 != count)) store_all(slot_c<0>());
        else store_all(slot_c<1>());
    };
    __builtin_amdgcn_s_waitcnt(0x0F70); // (all that was fetched so far is there: from here on the waits count)
    if (!works) { // fetches only
        auto help = [&](uint32_t t, auto slot_tag) __attribute__((always_inline)) {
            arrived(slot_c<(kSlots - 2) * kFetches>());
            fetch(t + kSlots - 1, slot_c<decltype(slot_tag)::value + kSlots - 1>());
        };
        for (uint32_t t = 0; t < count; t += kSlots) {
            help(t, slot_c<0>());
            if (t + 1 >= count) break;
            help(t + 1, slot_c<1>());
            if (t + 2 >= count) break;
            help(t + 2, slot_c<2>());
            if constexpr (kSlots > 3) {
                if (t + 3 >= count) break;
                help(t + 3, slot_c<3>());
            }
        }
    }
    else
        for (uint32_t t = 0; t < count; t += kSlots) {
            tile(t, slot_c<0>());
            if (t + 1 >= count) break;
            tile(t + 1, slot_c<1>());
            if (t + 2 >= count) break;
            tile(t + 2, slot_c<2>());
            if constexpr (kSlots > 3) {
                if (t + 3 >= count) break;
                tile(t + 3, slot_c<3>());
            }
        }
    __builtin_amdgcn_s_waitcnt(0x0F70); // (no fetch may outlive the workgroup's LDS)
}

struct TileConfig {
    int tm, tn;
};
// Index 0 is "choose for me"; 1.. are explicit (5: e2m3 only; 6: full grids only; 7: strips, dots_strips_kernel; 8 and 9: A in
// registers, dots_resident_kernel with one and two blocks of rows).
constexpr TileConfig kConfigs[] = {{0, 0}, {8, 2}, {4, 2}, {4, 1}, {2, 1}, {4, 4}, {1, 1}, {4, 2}, {4, 2}, {4, 2}};
constexpr int kConfigCount = sizeof(kConfigs) / sizeof(kConfigs[0]);
constexpr int kTriangleConfigs = 6; // the shapes below this index serve triangular grids


/** Tiles of a bm x bn grid over m x n outputs with something on or right of the diagonal col = row + shift. */
inline uint32_t log2_of(uint32_t power_of_two) { return (uint32_t)__builtin_ctz(power_of_two); }
inline uint64_t live_tiles(uint64_t m, uint64_t n, uint32_t bm, uint32_t bn, uint32_t shift) {
    uint32_t const tiles_m = (uint32_t)((m + bm - 1) / bm), tiles_n = (uint32_t)((n + bn - 1) / bn);
    uint64_t count = 0;
    for (uint32_t t = 0; t < tiles_m; ++t) {
        uint32_t const from = first_live_tile(t, log2_of(bm), log2_of(bn), shift);
        count += from < tiles_n ? tiles_n - from : 0;
    }
    return count;
}
inline size_t triangle_scratch_bytes(uint64_t m, uint64_t n, uint32_t bm, uint32_t bn, uint32_t shift) {
    return (size_t)live_tiles(m, n, bm, bn, shift) * 8;
}

/** Rows of A that the pipelined loop reads by shifted loads (see dots_packed_kernel). */
template <class T>
inline bool needs_shift(GemmArgs const &g) {
    return g.avec < (T::kSrcChunk < 4 ? T::kSrcChunk : 4) && g.k_chunks / kStageChunks >= 4;
}

/** A straight into LDS (see the kernel): the largest tile of the types that reach LDS as they are, depths of whole
 *  trips of four stages, and for the two-accumulator types folds that fall between trips (measured at 8192^3,
 *  alternating in one session: i8 0.438 -> 0.419 ms, bf16 0.930 -> 0.902, f16 0.997 -> 0.968; with a fold after every
 *  second stage of the trip instead, the compiler ran out of registers in the folds and bf16 took 1.10 ms). Of 128 x 128 the
 *  integers, from 24 stages and more than two rows of tiles on (486 shapes of i8, 0.965 of the time in the mean; going round twelve sets of
 *  operands 2048 x 2048 x 4096 37.0 and 35.9 us, x 3072 33.1 and 32.7, but x 2560 31.0 and 31.0 and x 2048 28.7 and 29.1). */
template <class T, int TM, int TN>
constexpr bool direct_built() {
    return kDirectStaging && !T::kUnsigned && !T::kPrewiden && T::kSrcChunk == 16 && T::kImageChunk == 16 &&
           ((TM == 8 && TN == 2) || (TM == 4 && TN == 1 && !T::kChunked) || (TM == 4 && TN == 2 && T::kChunked));
}
template <class T, int TM, int TN>
bool goes_direct(GemmArgs const &g) {
    if constexpr (!direct_built<T, TM, TN>()) return false;
    uint32_t const stages = g.k_chunks / kStageChunks;
    bool const whole = g.k_src_bytes % (2 * kStageChunks * T::kSrcChunk) == 0;
    return !needs_shift<T>(g) && g.metric == 0 && stages % 4 == 0 && stages >= 8 && (whole || !tail_matters_for<T, false>()) &&
           (!T::kChunked || g.chunk_stages % 4 == 0) && (TN == 2 || (stages >= 24 && g.m > 256)) && g.avec >= 16 &&
           !(forced_tile_config() & 0x40000000);
}

/** `slots_only`: do not launch, only report how many workgroups of the kernel this call would use are resident on
 *  the device at once. */
template <class T, int TM, int TN>
hipError_t launch_one(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle, int *slots_only = nullptr) {
    constexpr int BM = TM * 32, BN = TN * 128;
    g.tiles_m = (g.m + BM - 1) / BM;
    g.tiles_n = (g.n + BN - 1) / BN;
    uint64_t tiles = (uint64_t)g.tiles_m * g.tiles_n;
    if (tiles > 0x7FFFFFFFull) return hipErrorInvalidValue;
    g.tile_list = nullptr;
    if (triangle) {
        tiles = live_tiles(g.m, g.n, BM, BN, g.tri_shift);
        if (!tiles) return hipSuccess;
        if (triangle_scratch_bytes(g.m, g.n, BM, BN, g.tri_shift) > triangle->bytes) return hipErrorInvalidValue;
        g.tile_list = triangle->words;
    }
    g.tile_count = (uint32_t)tiles;
    // The tile's A offsets are 32-bit: (rows of a tile) * stride must stay below 4 GiB.
    if ((uint64_t)BM * g.a_stride + 8 > 0xFFFFFFFFull) return hipErrorInvalidValue;
    // So are the per-lane C offsets: 4 rows plus the tile's width.
    if (4 * (uint64_t)g.c_stride + BN * 4 > 0xFFFFFFFFull) return hipErrorInvalidValue;
    // The offsets into a wavefront's B tiles are 32-bit as well.
    if ((uint64_t)(TN + 1) * g.k_chunks * kTileRows * T::kImageChunk > 0xFFFFFFFFull) return hipErrorInvalidValue;
    // The pipeline runs across tile boundaries when the pipelined loop takes the stages of a tile (A readable
    // with dword loads, or shifted into place behind them: bf16 959 x 74,207 x 4307 took 5.6 ms in the guarded loop) and
    // there are enough of them to prefetch three ahead.
    uint32_t const stages = g.k_chunks / kStageChunks;
    bool const self = triangle && triangle->self && stages >= 4 && (uint64_t)TM * g.k_chunks * kTileRows * T::kImageChunk <= 0xFFFFFFFFull;
    bool const shifted = !self && needs_shift<T>(g);
    bool const across = !shifted && stages >= 4;
    bool const norms = g.metric != 0;
    // depths that fill an even number of stages exactly: the pipelined kernel without the tail masks
    bool const whole = across && g.k_src_bytes % (2 * kStageChunks * T::kSrcChunk) == 0;
    void (*kernel)(GemmArgs) = across ? dots_packed_kernel<T, TM, TN, true, false> : dots_packed_kernel<T, TM, TN, false, false>;
    if constexpr (TM * TN < 16) {
        if (shifted) kernel = dots_packed_kernel<T, TM, TN, true, false, false, false, true>;
    }
    else if (shifted) return hipErrorInvalidValue; // (launch_typed does not ask for it)
    if constexpr (tail_matters_for<T, false>()) {
        if (whole) kernel = dots_packed_kernel<T, TM, TN, true, false, true>;
    }
    bool direct = false;
    if constexpr (direct_built<T, TM, TN>()) {
        direct = goes_direct<T, TM, TN>(g);
        if (direct) kernel = dots_packed_kernel<T, TM, TN, true, false, tail_matters_for<T, false>(), true>;
    }
    if constexpr (T::kDistances) {
        if (norms) kernel = across ? dots_packed_kernel<T, TM, TN, true, true> : dots_packed_kernel<T, TM, TN, false, true>;
        if constexpr (TM * TN < 16) {
            if (norms && shifted) kernel = dots_packed_kernel<T, TM, TN, true, true, false, false, true>;
        }
        if (norms && whole) kernel = dots_packed_kernel<T, TM, TN, true, true, true>;
    }
    else if (norms) return hipErrorInvalidValue;
    // Shallow products of the two-accumulator types fold after every trip of the loop: no branch, and nothing to clear.
    bool folds = false;
    if constexpr (T::kChunked && !T::kDeepOnly && TM * TN > 1) {
        folds = !direct && !self && (across || shifted) && g.chunk_stages == 2;
        if (folds && !norms) kernel = shifted ? dots_packed_kernel<T, TM, TN, true, false, false, false, true, true>
                                      : whole ? dots_packed_kernel<T, TM, TN, true, false, true, false, false, true> : dots_packed_kernel<T, TM, TN, true, false, false, false, false, true>;
        if (folds && norms) kernel = shifted ? dots_packed_kernel<T, TM, TN, true, true, false, false, true, true>
                                     : whole ? dots_packed_kernel<T, TM, TN, true, true, true, false, false, true> : dots_packed_kernel<T, TM, TN, true, true, false, false, false, true>;
    }
    // All pairs: A from the image, where it lies as the MFMA wants it (widened, its rows' ends zero, its sums taken).
    if constexpr (TM * TN > 1 && TM * TN < 16 || (TM == 8 && TN == 2)) {
        constexpr bool kFolds = T::kChunked && !T::kDeepOnly;
        if (self) {
            direct = false;
            folds = kFolds && g.chunk_stages == 2;
            kernel = folds ? dots_packed_kernel<T, TM, TN, true, false, false, false, false, kFolds, true> : dots_packed_kernel<T, TM, TN, true, false, false, false, false, false, true>;
            if constexpr (T::kDistances) {
                if (norms) kernel = folds ? dots_packed_kernel<T, TM, TN, true, true, false, false, false, kFolds, true> : dots_packed_kernel<T, TM, TN, true, true, false, false, false, false, true>;
            }
        }
    }
    // Persistent grid: as many workgroups as fit on the device at once (queried once per kernel; threads that
    // ask at the same time store the same number).
    static std::atomic<int> resident_of[26];
    std::atomic<int> &slot = resident_of[self ? 22 + (norms ? 1 : 0) + (folds ? 2 : 0) : (shifted ? (norms ? 10 : 9) : direct ? 8 : (across ? 1 : 0) + (norms ? 2 : 0) + (whole ? 4 : 0)) + (folds ? 11 : 0)];
    int resident = slot.load(std::memory_order_relaxed);
    if (!resident) {
        int per_cu = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (void const *)kernel, 256, 0);
        if (e != hipSuccess) return e;
        int const units = compute_unit_count();
        resident = (per_cu > 0 ? per_cu : 1) * (units > 0 ? units : 256);
        slot.store(resident, std::memory_order_relaxed);
    }
    if (slots_only) {
        *slots_only = resident;
        return hipSuccess;
    }
    // Stores past the caches reach the memory as they are, and partial lines of two workgroups on a compute unit get in each other's way
    // where they are most of the work: 128 x 128 of the two-accumulator types, one and two of them (us): bf16 99,543 x 1482 x 320 213 and
    // 287, 1,000,000 x 130 x 768 598 and 716, e4m3 101,986 x 1059 x 512 179 and 211; the mean of fourteen such shapes 0.83. Of
    // 17 to 31 stages two are faster again (seventeen shapes, 0.93).
    if (T::kChunked && TM * TN == 4 && g.store_policy == 1 && stages <= 16 && compute_unit_count() > 0 && resident > compute_unit_count()) resident = compute_unit_count();
    uint32_t const blocks = (uint32_t)(tiles < (uint64_t)resident ? tiles : (uint64_t)resident);
    // Shallow products with several tiles per workgroup are bound by their stores: spread the starts over about the
    // time one round of tiles takes to store (the chip writes some 5.5 TB/s in this pattern; ticks of 10 ns).
    g.stagger_ticks = 0;
    if (stages <= 16 && tiles >= 4 * (uint64_t)blocks) {
        double const round_bytes = (double)BM * BN * 4 * blocks;
        g.stagger_ticks = (uint32_t)(round_bytes / 5.5e12 * 1e8);
    }
    int const forced = forced_tile_config();
    if ((forced >> 8) & 0xFFFFF) g.stagger_ticks = (uint32_t)((forced >> 8) & 0xFFFFF) - 1; // (test hook: bits 8..27 = ticks + 1)
    if ((forced >> 28) & 3) g.store_policy = (uint32_t)(forced >> 28) & 3;                  // (test hook: bits 28..29)
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, g);
    return hipGetLastError();
}

/** LDS of dots_strips_kernel. */
constexpr size_t strips_lds_bytes(int bm, int batch, uint32_t stages) {
    return (size_t)stages * bm * kStageBytes + (size_t)batch * kStripColumns * 4 + (size_t)bm * (32 + 3) * 4;
}
constexpr size_t kStripsLds = 160 << 10;
template <class T>
inline bool strips_possible(GemmArgs const &g) {
    uint32_t const stages = g.k_chunks / kStageChunks;
    return stages >= 2 && strips_lds_bytes(64, 16, stages) <= kStripsLds && (!T::kChunked || g.chunk_stages == 2) && g.n >= 128 &&
           g.c_stride >= 4 * (uint64_t)g.n && g.c_stride < (1u << 24) - 1024;
}
/** How many strips each row of tiles is cut into: of the numbers that fill whole rounds of resident workgroups, the one whose rounds
 *  walk the fewest tiles, a tile's worth for starting and ending each strip included. Eight candidates, each the most strips that
 *  fit the rounds they need (fewer walk as far); trying every number up to several hundred took 2.8 us of a call with few rows. */
struct StripPlan {
    uint32_t tiles_m, strips, strip_tiles;
};
inline StripPlan strip_plan(uint32_t m, uint32_t n, uint32_t bm) {
    uint64_t const resident = compute_unit_count() > 0 ? compute_unit_count() : 256; // (one workgroup's registers fill a compute unit)
    uint64_t const tiles_m = (m + (uint64_t)bm - 1) / bm, tiles = ((uint64_t)n + kStripColumns - 1) / kStripColumns;
    uint64_t best = ~0ull, length = tiles;
    uint64_t strips = 1;
    for (int candidate = 0; candidate < 8; ++candidate) {
        uint64_t const rounds = (tiles_m * strips + resident - 1) / resident;
        strips = rounds * resident / tiles_m;
        uint64_t const here = strips < tiles ? (tiles + strips - 1) / strips : 1;
        if (rounds * (here + 1) < best) best = rounds * (here + 1), length = here;
        if (here == 1) break;
        ++strips;
    }
    return {(uint32_t)tiles_m, (uint32_t)((tiles + length - 1) / length), (uint32_t)length};
}
template <class T, int TM, int BATCH>
hipError_t launch_strips_as(GemmArgs &g, hipStream_t stream, PlannedTile *planned) {
    constexpr int BM = TM * 32;
    void (*kernel)(GemmArgs) = dots_strips_kernel<T, TM, 0, BATCH>;
    if constexpr (T::kDistances) {
        if (g.metric == 1) kernel = dots_strips_kernel<T, TM, 1, BATCH>;
        if (g.metric == 2) kernel = dots_strips_kernel<T, TM, 2, BATCH>;
    }
    else if (g.metric != 0) return hipErrorInvalidValue;
    StripPlan const plan = strip_plan(g.m, g.n, BM);
    g.tiles_m = plan.tiles_m, g.tiles_n = plan.strips, g.strip_tiles = plan.strip_tiles;
    uint64_t const units = (uint64_t)g.tiles_m * g.tiles_n;
    if (units > 0x7FFFFFFFull) return hipErrorInvalidValue;
    if (planned) {
        planned->shape = 7, planned->units = (uint32_t)units, planned->strip_tiles = g.strip_tiles;
        return hipSuccess;
    }
    g.tile_count = (uint32_t)units, g.tile_list = nullptr;
    uint64_t const resident = compute_unit_count() > 0 ? compute_unit_count() : 256;
    hipLaunchKernelGGL(kernel, dim3((uint32_t)(units < resident ? units : resident)), dim3(64 * kStripWaves),
                       strips_lds_bytes(BM, BATCH, g.k_chunks / kStageChunks), stream, g);
    return hipGetLastError();
}
/** Rows of a strip: 128 up to six stages, 64 beyond and for few rows. */
inline uint32_t strip_rows(uint32_t m, uint32_t stages) { return m > 64 && strips_lds_bytes(128, 32, stages) <= kStripsLds ? 128 : 64; }
template <class T>
hipError_t launch_strips(GemmArgs &g, hipStream_t stream, PlannedTile *planned) {
    return strip_rows(g.m, g.k_chunks / kStageChunks) == 128 ? launch_strips_as<T, 4, 32>(g, stream, planned) : launch_strips_as<T, 2, 16>(g, stream, planned);
}

/** Which of these kernels there are. Left out are those whose registers do not fit (two-accumulator types of 12 stages; of 10 with
 *  the angular finaliser; two blocks of rows beside anything but a plain store): a reload in the loop would wait for the stores in front
 *  of it. None is left that has any there (u8 dots of 10 stages off the lines and u8 angular of 12 save one register around the loading
 *  of A). Or those that were slower than strips: rows off the lines of up to four stages (i8
 *  1000 x 500,009 x 301 550 and 571) and the angular finaliser there (two-accumulator types only at 8 stages, integers from 8 on), or on lines
 *  with an integer loop of two stages. */
template <class T, int TM, int STAGES, int METRIC, bool CARRY>
constexpr bool resident_built() {
    if (T::kImageChunk != 16 || T::kDeepOnly || (METRIC != 0 && !T::kDistances) || STAGES % 2 != 0 || STAGES > (T::kChunked ? 10 : 12)) return false;
    if (TM == 2) return METRIC == 0 && !CARRY && STAGES <= (T::kChunked ? 4 : 6);
    if (METRIC == 1 && (T::kChunked ? STAGES > 8 : STAGES < 4)) return false;
    return !CARRY || (STAGES >= (METRIC == 1 ? 8 : 6) && STAGES <= 10);
}
typedef void (*resident_kernel_t)(GemmArgs);
template <class T, int TM, int METRIC, bool CARRY, int STAGES = 2>
resident_kernel_t resident_kernel_of(uint32_t stages) {
    if constexpr (STAGES > 12) return nullptr;
    else {
        if (stages != STAGES) return resident_kernel_of<T, TM, METRIC, CARRY, STAGES + 2>(stages);
        if constexpr (resident_built<T, TM, STAGES, METRIC, CARRY>()) return dots_resident_kernel<T, TM, STAGES, METRIC, CARRY>;
        else return nullptr;
    }
}
/** The kernel for these arguments with `tm` blocks of 32 rows per wavefront (1 or 2); NULL: there is none. */
template <class T>
resident_kernel_t resident_kernel(GemmArgs const &g, int tm) {
    uint32_t const stages = g.k_chunks / kStageChunks;
    bool const lines = (((uintptr_t)g.c | g.c_stride) & 127) == 0;
    // (a wavefront's rows of A and of C lie within 31 bits; the two-accumulator types' sums go into their totals every two stages)
    if (g.c_stride < 4 * (uint64_t)g.n || g.c_stride >= (1u << 24) || g.a_stride >= (1u << 24) - 1 || (T::kChunked && g.chunk_stages != 2)) return nullptr;
    if (tm == 2) return lines && g.metric == 0 ? resident_kernel_of<T, 2, 0, false>(stages) : nullptr;
    switch (g.metric) {
    case 0: return lines ? resident_kernel_of<T, 1, 0, false>(stages) : resident_kernel_of<T, 1, 0, true>(stages);
    case 1: return lines ? resident_kernel_of<T, 1, 1, false>(stages) : resident_kernel_of<T, 1, 1, true>(stages);
    default: return lines ? resident_kernel_of<T, 1, 2, false>(stages) : resident_kernel_of<T, 1, 2, true>(stages);
    }
}
/** Rows are shared out evenly over as few workgroups as hold them, and the columns are cut into strips so that whole rounds of
 *  workgroups (one per compute unit) walk the fewest tiles, four to each strip for its start: as strip_plan.
 *
 *  `in_step`: where rows of C are a multiple of 4 KiB apart and strips too (32 tiles of 32 columns), all workgroups, which go at about the same
 *  pace, write to addresses that agree in their lower twelve bits all the time, and those share few of the memory's channels (i8 4982 x
 *  12,288 x 256 72.5 us, 50.7 through tiles). Up to 24 workgroups of rows a strip of 32 to 128 tiles has one more then: the time of 32 is 0.93
 *  in the mean of 770 dots, 0.94 of 414 euclidean and 0.98 of 274 angular, of 128 0.95, 0.94 and 0.97. With more rows that does not help (0.98
 *  to 1.02), nor do longer strips gain (0.97 to 1.0, 1.0 and 1.0 to 1.02; 1024 x 1,048,576 x 768 1082 us and 1086). */
struct ResidentPlan {
    uint32_t blocks, waves, strips, strip_tiles;
    bool in_step;
};
inline ResidentPlan resident_plan(uint32_t m, uint32_t n_tiles, uint32_t bm, uint64_t c_stride) {
    uint64_t const resident = compute_unit_count() > 0 ? compute_unit_count() : 256, rows = kResidentWaves * (uint64_t)bm;
    uint64_t const least = (m + rows - 1) / rows, waves = ((m + least - 1) / least + bm - 1) / bm, blocks = (m + waves * bm - 1) / (waves * bm);
    uint64_t best = ~0ull, length = n_tiles, strips = 1;
    for (int candidate = 0; candidate < 8; ++candidate) {
        uint64_t const rounds = (blocks * strips + resident - 1) / resident;
        strips = rounds * resident / blocks;
        uint64_t const here = strips < n_tiles ? (n_tiles + strips - 1) / strips : 1;
        if (rounds * (here + 4) < best) best = rounds * (here + 4), length = here;
        if (here == 1) break;
        ++strips;
    }
    bool const in_step = c_stride % 4096 == 0 && length % 32 == 0;
    if (in_step && blocks <= 24 && length <= 128 && length < n_tiles) ++length;
    return {(uint32_t)blocks, (uint32_t)waves, (uint32_t)((n_tiles + length - 1) / length), (uint32_t)length, in_step};
}
/** `planned`: nothing is launched. */
template <class T>
hipError_t launch_resident(GemmArgs &g, hipStream_t stream, int tm, PlannedTile *planned) {
    resident_kernel_t const kernel = resident_kernel<T>(g, tm);
    if (!kernel) return hipErrorInvalidValue;
    ResidentPlan const plan = resident_plan(g.m, g.n_tiles, 32 * tm, g.c_stride);
    uint64_t const units = (uint64_t)plan.blocks * plan.strips;
    if (units > 0x7FFFFFFFull) return hipErrorInvalidValue;
    if (planned) {
        planned->resident_rows = 32 * tm, planned->resident_units = (uint32_t)units, planned->resident_tiles = plan.strip_tiles;
        return hipSuccess;
    }
    g.tiles_m = plan.blocks, g.tiles_n = plan.strips, g.strip_tiles = plan.strip_tiles, g.strip_waves = plan.waves;
    g.tile_count = (uint32_t)units, g.tile_list = nullptr;
    hipLaunchKernelGGL(kernel, dim3((uint32_t)units), dim3(64 * kResidentWaves), 0, stream, g);
    return hipGetLastError();
}

template <class T>
hipError_t launch_config(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle, int config,
                         int *slots_only = nullptr) {
    switch (config) {
    case 1:
        if constexpr (T::kChunked) return hipErrorInvalidValue;
        else return launch_one<T, 8, 2>(g, stream, triangle, slots_only);
    case 2: return launch_one<T, 4, 2>(g, stream, triangle, slots_only);
    case 3: return launch_one<T, 4, 1>(g, stream, triangle, slots_only);
    case 5:
        if constexpr (T::kDtype != kE2M3) return hipErrorInvalidValue;
        else return launch_one<T, 4, 4>(g, stream, triangle, slots_only);
    case 6:
        if (triangle) return hipErrorInvalidValue; // (launch_typed does not ask for it)
        return launch_one<T, 1, 1>(g, stream, nullptr, slots_only);
    default: return launch_one<T, 2, 1>(g, stream, triangle, slots_only);
    }
}

template <class T>
hipError_t launch_typed(GemmArgs &g, hipStream_t stream, TriangleScratch const *triangle) {
    int const forced = forced_tile_config();
    int config = forced & 0x7F;
    bool const chosen_here = config <= 0 || config >= kConfigCount;
    PlannedTile *const planned = forced < 0 ? planned_tile() : nullptr;
    auto tiles_of = [&](GemmArgs const &args, int c) {
        uint64_t const bm = kConfigs[c].tm * 32, bn = (uint64_t)kConfigs[c].tn * 128;
        if (triangle) return live_tiles(args.m, args.n, (uint32_t)bm, (uint32_t)bn, args.tri_shift);
        return ((args.m + bm - 1) / bm) * ((args.n + bn - 1) / bn);
    };
    auto unaligned_rows_of_c = [&](GemmArgs const &args) { return !triangle && args.metric == 0 && (((uintptr_t)args.c | args.c_stride) & 127) != 0; };
    // (strides that the 32-bit offsets of a taller or wider tile could not span stay with the small one)
    auto roomy = [](GemmArgs const &args) { return args.m >= 128 && args.a_stride < (1u << 24) - 1 && args.c_stride < (1u << 30) - 1024; };
    struct Choice {
        int config;
        uint32_t store_policy;
        Choice(int config, uint32_t store_policy = 0) : config(config), store_policy(store_policy) {}
    };
    auto past = [](int config) { return Choice(config, 1); };
    // Strips (see dots_strips_kernel) where C is large against the operands. What they save is the partial lines of rows off the lines
    // and the staging of A with every tile; what they cost is the start and the end of every strip, with nothing beside it on the
    // compute unit, and the columns of a row's last tile. (Calls that keep A in registers, resident_blocks, do not ask here. Of dots on lines that
    // leaves u1, short ones whose strips would write in step, and rows of A 16 MiB apart; times of other dots on lines in this comment and the next are of what they
    // would take without it, and the choice is that too.) So a row of C has to be more than eight tiles of 256 columns and a strip at
    // least four, or three where what the tiles do besides their columns is more (distances; e2m3, which widens: 2038 x 10,937 x 77 43 us
    // and 113, u4 angular 436 x 39,391 x 122 55 and 90; of 240 such shapes two in a hundred were slower): with fewer they took up to twice as long as the tiles below, now and before (us): i8 1,000,000 x 130 x 768 638
    // and 447, angular 817 and 482; bf16 200,000 x 129 x 768 227 and 152; u8 714 x 25,854 x 198 (three to a strip) 31 and 26. On
    // lines there are no partial ones to save, and a row has to be 32,768 long: i8 euclidean 349,434 x 448 x 64 279 and 151, 6718 x
    // 20,000 x 448 172 and 150; two stages also take 512 MiB (u4 947 x 85,152 x 64 75 and 67). Deep distances of the types whose tiles
    // widen A or sum its bytes: 8192 (e2m3 angular 14,922 x 18,880 x 2041 715 and 1073, u4 angular 1.19 times as fast in the mean of
    // 110 shapes; of i8 and of u8 euclidean half of the shapes would lose by it).
    // Two dot products of integers do not gain by whole lines: deep ones into rows on the memory's sectors, whose partial lines cost it
    // little (i4 3276 x 27,600 x 1920 267 and 210; not e2m3, whose tiles widen: 1.15 to 1.29 times as fast as strips in the mean of 700
    // such shapes), and those that take two strips of 64 rows where one tile of 128 holds all
    // rows of A and reads the image once (u8 angular 109 x 242,980 x 1792 156 and 138). Nor do those of little work, two stages into a C
    // that the last-level cache takes in (u1 135 x 138,111 x 98 46 and 35, i4 5384 x 4087 x 212 48 and 38, bf16 5377 x 4053 x 29 47 and
    // 39; of 900 such shapes up to 96 MiB, 112 of the narrow types, half were slower). The 4-bit types' tiles stage half of the bytes: not
    // deep ones whose image no cache holds and every 64 rows would read again (u4 1239 x 188,257 x 1567 741 and 555), and on lines
    // none below 512 MiB (u4 793 x 137,216 x 317 142 and 116) or of two stages (u4 161 x 1,191,936 x 75 265 and 238, u1 640 x 212,864 x 55 136
    // and 130). The bytes' rows on 16 bytes, deep, with an image under 100 MiB: 0.95 of the time before as tiles in the mean of 34.
    auto strips_pay = [&](GemmArgs const &args, bool lines, uint64_t mib) -> bool {
        if constexpr (T::kDeepOnly) return false;
        uint32_t const stages = args.k_chunks / kStageChunks;
        bool const norms = args.metric != 0, nibbles = T::kDtype == kI4 || T::kDtype == kU4;
        if (!strips_possible<T>(args) || stages > 16 || args.n <= 2048) return false;
        if (lines) {
            bool const wide_terms = norms && stages > 8 && (nibbles || T::kDtype == kE2M3 || (T::kDtype == kU8 && args.metric == 1));
            if (args.m <= 64 || mib < (norms || (stages > 2 && !nibbles) ? 256 : 512) || args.n < (wide_terms ? 8192u : 32768u)) return false;
            if (!norms && stages <= 2 && (nibbles || T::kDtype == kU1)) return false;
            if (T::kChunked ? !norms && stages > 8 : norms ? stages > 2 && stages <= 8 && (stages > 4 || mib < 512) : stages > 4) return false;
        }
        else {
            if (mib < (stages > 2 ? 96 : norms || T::kDtype == kE2M3 ? 64 : nibbles || T::kDtype == kU1 ? 112 : 96)) return false;
            uintptr_t const rows_at = (uintptr_t)args.c | args.c_stride;
            uint64_t const image_mib = ((uint64_t)args.n_tiles * args.k_chunks * kTileRows * T::kImageChunk) >> 20;
            uintptr_t const sector = (T::kDtype == kI8 || T::kDtype == kU8) && image_mib < 100 ? 15 : 31;
            if (!T::kChunked && T::kDtype != kE2M3 && !norms && ((stages > 8 && ((rows_at & sector) == 0 || (nibbles && image_mib >= 256))) || (stages > 4 && (rows_at & 63) == 0))) return false;
            if (!T::kChunked && args.m > 64 && args.m <= 128 && strip_rows(args.m, stages) == 64) return false;
        }
        return strip_plan(args.m, args.n, strip_rows(args.m, stages)).strip_tiles >= (norms || T::kDtype == kE2M3 ? 3 : 4);
    };
    // Where storing C is most of the work, what counts is how much of it there is, against the 256 MiB of the last-level
    // cache above all, and whether its rows start on lines. Drawn through 980 random shapes (33 to 8192 rows, depths of 1 to 64
    // stages, C of 4 to 2200 MiB, half of them with rows off the lines; whole calls that go round three sets of operands and
    // results), every tile and the strips at each, and again through 3000 with up to 2.5 million rows. Some of them (us, before and
    // now): u8 euclidean 1000 x 500,009 x 301 1165 and 610 (strips), i8 1024 x 204,801 x 220 298 and 151 (strips), f16 8192 x 8191 x
    // 1000 289 and 230 (strips); with rows on
    // lines bf16 208 x 60,160 x 485 71 and 43 (64 x 128), e5m2 150 x 136,704 x 320 84 and 63 (64 x 128), i8 angular 371 x
    // 34,739 x 1600 154 and 58 (64 x 128), bf16 527 x 400,384 x 192 384 and 259 (strips; 228 with A in registers), bf16 3439 x 38,656 x 826 382 and 316
    // (128 x 128: two workgroups of it fit a compute unit, and the kernels for depths of no whole stage spill at 128 x 256).
    // 0: nothing here applies.
    auto by_bytes_of_c = [&](GemmArgs const &args) -> int {
        uint32_t const stages = args.k_chunks / kStageChunks;
        uint64_t const mib = ((uint64_t)args.m * args.n * 4) >> 20;
        bool const lines = (((uintptr_t)args.c | args.c_stride) & 127) == 0, norms = args.metric != 0;
        bool const whole = args.k_src_bytes % (2 * kStageChunks * T::kSrcChunk) == 0, nibbles = T::kDtype == kI4 || T::kDtype == kU4;
        if (strips_pay(args, lines, mib)) return 7;
        if (args.m <= 64) return 0;
        // Two tiles of 64 rows read the image twice, which is most of a deep product of few rows (u4 74 x 178,464 x 1664 89 us and 76
        // through 128 x 128, i8 angular 79 x 269,824 x 2122 207 and 168).
        if (!T::kChunked && args.m <= 128 && stages > (norms ? 16 : 4)) return 0;
        // Three tiles of 64 rows, but four of them in two of 128: 128 x 128 gains nothing by its second workgroup there (e5m2 angular 133 x
        // 1,285,455 x 3780 4683 us and 3272 before it, bf16 euclidean 133 x 419,427 x 2376 1073 and 830, f16 angular 192 x 252,615 x 1731
        // 481 and 461) but for deep rows into a middling C off the lines (1.1 times as fast).
        if (T::kChunked && norms && args.m > 128 && args.m <= 192 && (lines || stages < 32 || mib >= 300 || args.m <= 144)) return 0;
        if (!lines) {
            // (Shallow products into so large a C belong to strips or, where those do not pay, to the rule at the end.)
            if (stages <= 16 && mib >= (stages <= 2 ? 64 : 96)) return 0;
            // Depths at which the MFMAs are most of the work again: the largest tiles, once there are enough of them (e2m3 euclidean
            // 78,940 x 2733 x 12,009 5265 through 128 x 128 and 3664 through 256 x 256, f16 5825 x 48,330 x 5312 4360 and 4006; dots
            // e4m3 755 x 53,520 x 5376 458 and 425).
            // How deep those begin was timed at 2000 shapes, 128 x 128 against the largest tile: e2m3, whose largest is 128 x 512, 0.89
            // of its time at 24 to 32 stages into 256 MiB and more, u4 1.18 and 1.05 up to 60; of the 8-bit floats into rows that
            // start on odd words 1.05 to 1.16 up to 90 (into rows on halves of lines e4m3 755 x 53,520 x 5376 as above), bf16 0.95, dots 1.04 to 1.12.
            bool const odd_rows = (((uintptr_t)args.c | args.c_stride) & 7) != 0;
            if (norms && !T::kChunked) {
                if (stages <= 16 || mib < 32) return 4;
                uint32_t const deepest = T::kDtype == kE2M3 ? (mib < 256 ? 40 : 16) : mib < 256 || T::kDtype == kU4 ? 60 : 32;
                return stages <= deepest ? 3 : 0;
            }
            uint32_t const deepest = odd_rows && (!norms || T::kDtype == kE4M3 || T::kDtype == kE5M2) ? 90 : 60;
            if (norms) return stages > 16 && mib >= 96 && (stages <= deepest || mib < 300) ? 3 : 0;
            if (T::kChunked) return mib >= 32 && ((stages > 4 && mib < 96) || (stages > 16 && mib < 256)) && stages <= deepest ? 3 : 0;
            return stages <= 16 && mib < 96 ? 4 : 0;
        }
        // (two columns of tiles: A is read twice by the small ones; i8 216,199 x 256 x 384 94 and 62 through 256 x 256)
        if (!T::kChunked && args.n <= 256 && mib >= 128) return 0;
        if (T::kChunked && norms) return stages > 16 && stages < 32 && mib >= 64 ? 3 : 0;
        if (T::kChunked) {
            if (mib < 96) return stages > 2 && (stages <= 16 || (stages < 32 && !whole)) ? 4 : 0;
            if (stages <= 2) return 0;
            if (stages <= 4 && mib < 256) return 4;
            return stages <= 16 || (stages < 32 && !whole) ? 3 : 0; // (f16 4542 x 16,384 x 324, which keeps A in registers now, 113 us, 167 through the largest tile)
        }
        if (!norms) {
            if (stages > 16) return 0;
            if (mib < 96) return stages <= 8 || mib >= 32 ? 4 : 0; // (i8 2048^3 28.0 us through 128 x 128, 28.8 through 64 x 128)
            if (stages <= 4) return stages <= 2 ? 0 : mib < 256 || T::kDtype == kE2M3 ? 4 : 3;
            // (e2m3's 128 x 512 tile, and 256 x 256 of the bytes, are as fast or faster: e2m3 409 x 197,504 x 960 221 us through 128 x 128, 207)
            return stages <= 8 && mib < (nibbles || T::kDtype == kU1 ? 512 : T::kDtype == kE2M3 ? 130 : 200) ? 3 : 0;
        }
        if (stages > 16) return stages < 32 && mib < 96 ? 4 : 0;
        if (mib < 256) return stages <= 8 || mib < 96 ? 4 : 3;
        return stages > 2 && stages <= 4 && mib < 512 ? 4 : 0;
    };
    // All pairs, once A comes out of the image: drawn through 110 random shapes (256 to 16,384 vectors of 64 to 8192 values),
    // every tile at each. Some of them (us, the largest tile that fills the device and the one taken): dots i8 8192 x 768 81 and 63
    // (128 x 128), u8 11,269 x 320 188 and 122 (128 x 128), f16 4096 x 300 43 and 34 (64 x 128), e4m3 8192 x 1024 113 and 101 (128 x
    // 128); euclidean u4 13,649 x 1449 382 and 233 (128 x 128), e5m2 15,409 x 1216 447 and 365 (128 x 128); angular i8 8192 x 768 76
    // and 69 (64 x 128). 0: nothing here applies.
    auto by_tiles_of_triangle = [&](GemmArgs const &args) -> int {
        uint32_t const stages = args.k_chunks / kStageChunks;
        uint64_t const tiles = tiles_of(args, 3);
        bool const norms = args.metric != 0;
        if (T::kChunked && norms) return stages >= 12 && tiles >= 1500 ? 3 : 0;
        if (T::kChunked) {
            if (stages <= 2) return 0;
            if (stages < 32) return tiles >= 1024 ? 3 : tiles >= 256 ? 4 : 0;
            return tiles >= 512 && tiles < 1024 ? 3 : 0;
        }
        if (norms) return tiles < 600 ? 0 : stages <= 8 ? 4 : 3;
        return stages > 2 && tiles >= 1500 && (stages <= 16 || (T::kDtype == kU1 && stages <= 32)) ? 3 : 0;
    };
    // Largest tile that still gives every one of the 256 CUs at least one workgroup.
    auto choose = [&](GemmArgs const &args, int first) -> Choice {
        uint32_t const depth_stages = args.k_chunks / kStageChunks;
        // Few rows: a tile of more rows than A has multiplies what is not there (i8 1 x 1,048,576 x 768 through the 256-row
        // tile was bound by its matrix instructions), and one that is not full stores through the masked copy of the
        // epilogue. Measured, whole calls, the tile taken before against this one (us): i8 x 1,048,576 x 768 with 1 row 365
        // against 156 (32 x 128; 162 with 64 x 128), 32 rows 363 against 199, 64 rows 370 against 223 (64 x 128; 244 with
        // 32 x 128), 96 rows 391 against 261 (128 x 128); angular, 96 rows 351 against 275; bf16 1 row 361 against 288, 64
        // rows 399 against 376, 96 rows 442 against 426.
        if (!triangle && args.m <= 32) return 6;
        if (!triangle && args.m <= 64) first = 4;
        else if (!triangle && args.m < 128 && first < 3) first = 3;
        int best = 4;
        for (int c = first; c <= 4; ++c)
            if (tiles_of(args, c) >= 256) {
                best = c;
                break;
            }
        // Fewer tiles of 64 x 128 than CUs: 32 x 128 spreads the epilogues over more of them, which is most of a shallow
        // product's time (192 x 10,000 x 256, us: i8 angular 25.6 against 23.6, bf16 24.2 against 23.2, bf16 angular 28.1
        // against 25.2); a deep one gains as long as the smaller tiles fit one round (bf16 1024^3 26.3 against 24.8, angular
        // 29.3 against 26.1, but 64 x 30,000 x 4096 54 against 62).
        if (!triangle && tiles_of(args, 4) < 256 && (depth_stages <= 8 || tiles_of(args, 6) <= 256)) return 6;
        if (triangle && triangle->self && args.a_stride < (1u << 24) - 1 && args.c_stride < (1u << 30) - 1024)
            if (int const config = by_tiles_of_triangle(args); config >= first) return config;
        if (!triangle && args.a_stride < (1u << 24) - 1 && args.c_stride < (1u << 30) - 1024)
            if (int const config = by_bytes_of_c(args); config == 7 || (config && tiles_of(args, config) >= 256)) return config;
        // Distances over a shallow depth are bound by the epilogue (a finaliser and a store per output): two
        // workgroups per CU of 128 x 128 tiles overlap it with the other's loop better than one large tile does
        // (measured on 1024 x 1,048,576 x 768: 2.17 against 2.33 ms angular, 1.98 against 2.07 ms euclidean).
        // Since then the angular finaliser has become cheap where the cosine is small, and what is left of an epilogue's
        // cost is its length: the code of TM x TN x 16 finalisers and stores does not fit the instruction cache for the
        // large tiles. Measured, shallow depths (best shape against the others, ms): i8 angular 1024 x 1,048,576 x 768
        // 128 x 256 1.73, 256 x 256 1.78, 128 x 128 1.90, 64 x 128 2.09, but 8192 x 131,072 x 768 and 8192 x 8192 x
        // 1024 128 x 128 (1.42 against 1.55; 0.114 against 0.120); u8 128 x 128 (2.29 against 2.54 and 2.91); bf16
        // angular 1024 x 524,288 x 768 64 x 128 1.58 against 1.72 (128 x 128) and 2.18 (128 x 256), 8192 x 8192 x 1024
        // 0.198 against 0.267 and 0.319, and still 3.39 against 3.77 at depth 2048; f16 and e4m3 likewise.
        if (args.metric != 0 && T::kChunked) {
            if (depth_stages <= 32 && tiles_of(args, 4) >= 256) best = 4;
        }
        else if (args.metric != 0 && depth_stages <= 8) {
            if (!T::kUnsigned && args.m <= 2048 && best < 2 && tiles_of(args, 2) >= 256) best = 2;
            else if (best < 3 && tiles_of(args, 3) >= 256) best = 3;
        }
        // Two accumulator sets do not fit the 256 x 256 tile, and neither do the fifth dwords of shifted loads (99 registers
        // of the i8 kernel spill). In the 128 x 256 tile they cost the integers nothing; of the types with two accumulator
        // sets 37 to 68 registers spill there, where the kernels for aligned ragged rows spill 0 to 58.
        if ((T::kChunked || needs_shift<T>(args)) && best == 1) best = 2;
        // Two stages: the pipeline starts anew with every tile, the large tiles' kernels spill around that (e4m3 and e5m2 80
        // registers at 128 x 256, 13 before they held a loop for odd rows), and the stores are nearly all of the work. Measured,
        // the largest tile against 64 x 128 (us), C on whole lines: e4m3 2000 x 262,144 x 128 878 (767 with 13 spilled) against 424,
        // 1000 x 100,000 x 128 186 against 90, 300 x 60,000 x 128 33 against 18, 8192 x 8192 x 128 62 against 55; bf16 1130, 236, 39
        // and 67 against 430, 92, 20 and 57; i8 1228, 278, 41 and 71 against 414, 87, 18 and 51; the others likewise. Not the
        // floats up to 128 MiB of C in rows that are 64 KiB or a multiple apart (512 x 65,536 x 128, e4m3 32.8 against 34.2, bf16 35.6
        // against 36.2).
        if (depth_stages <= 2 && args.metric == 0 && args.m >= 128 && !unaligned_rows_of_c(args) &&
            !(T::kChunked && (args.c_stride & 0xFFFF) == 0 && (uint64_t)args.m * args.n * 4 <= 128ull << 20))
            return tiles_of(args, 4) >= 256 ? 4 : best;
        // e2m3 pays 13 vector operations for every dword of A it stages: a 128 x 512 tile (every wavefront 128 x 128)
        // stages half as much A per MFMA as 256 x 256 (8192^3: 0.51 against 0.59 ms; for i8 itself the two are equal). Rows of C
        // off the lines keep it: the rule below is of mixed use there (1000 x 300,009 x 304 579 against 813 us, but 512 x 153,601
        // x 900 240 against 186).
        // (not the f16 route of very deep rows: its two accumulator sets do not fit that tile)
        if (T::kDtype == kE2M3 && !T::kChunked && !triangle && args.metric == 0 && first == 1 && !needs_shift<T>(args) && tiles_of(args, 5) >= 256) return 5;
        // Products into rows of C that do not start on 128-byte lines. The stores of shallow ones go through the L2 (see the
        // epilogue) and take long enough to matter, and three small workgroups per compute unit overlap one's stores
        // with the others' loops, which one large tile cannot (measured, 64 x 128 against the tile chosen above: i8
        // 8192 x 8191 x 1000 0.129 against 0.142 ms, x 512 0.085 against 0.101; f16 8192 x 8191 x 1000 0.239 against
        // 0.280; i8 4096 x 4095 x 1000 0.036 against 0.039; deeper products and aligned rows lose by it).
        // That holds while the last-level cache (256 MiB) takes most of C in. A larger C is bound by the memory, which the small
        // tile's many short writes reach as they are, and what is best then depends on the image: as long as the cache can hold
        // that, C is better written past it. The lines below were drawn through 8700 timed shapes (128 to 8192 rows, C of 130
        // to 1700 MiB, depths to 2048, rows off the lines by 4 to 64 bytes; 5000 of them at random, every tile at each). The
        // time of 64 x 128 (of the largest tile for the deeper products) over that of the tile taken, mean and least: floats of 5
        // to 16 stages 1.22 and 0.79, deeper 1.08 and 0.85; integers of 2 stages 1.09 and 0.80, of 3 and 4 1.22 and 0.96, of 5
        // to 8 1.32 and 0.90, deeper 1.15 and 0.80 (16 in 1000 of all shapes lose more than 3 per cent); of the best tile at
        // each, 0.96. Those launches wrote the same C over and over; going round three sets of operands and results, 8000 random
        // shapes, the mean is 1.06 and 23 in 1000 lose more than 3 per cent. Most of those that it was drawn for go through strips now. What
        // is left comes here (see strips_pay): rows of C of up to 2048 columns, more than 16 stages, rows 16 MiB or more apart, and
        // the integers' rows on sectors. Some of them (us, 64 x 128 and what is taken): bf16 99,543 x 1482 x 320 387 and 236 (128 x 128 past
        // the caches, 322 through them), 2400 x 45,857 x 1500 654 and 523 (the same; 611 through 128 x 256, whose kernel for ragged depths of
        // 16-bit floats and for shifted rows spills), i8 2000 x 100,001 x 3000 1153 and 841 (256 x 256), 1,000,000 x 130 x 768 548 and 465 (128 x
        // 128 past the caches). Of many rows of few columns it is not always the best: i8 200,003 x 1001 x 304 372, 319 through 128 x 256.
        uint32_t const limit = T::kChunked ? 16 : 8;
        if (unaligned_rows_of_c(args) && best < 4 && depth_stages <= 2 * limit) {
            bool const shallow = depth_stages <= limit, bits = T::kDtype == kU1;
            Choice const small = tiles_of(args, 4) >= 256 ? 4 : best; // 64 x 128 where it gives every CU a tile
            uint64_t const c_mib = ((uint64_t)args.m * args.n * 4) >> 20;
            uint64_t const image_mib = ((uint64_t)args.n_tiles * args.k_chunks * kTileRows * T::kImageChunk) >> 20;
            uintptr_t const rows_at = (uintptr_t)args.c | args.c_stride;
            bool const halves = (rows_at & 63) == 0 && image_mib < 256; // rows on halves of lines: past the caches they cost no more than whole lines
            if (!roomy(args) || c_mib < 128) return shallow ? small : Choice(best);
            if (T::kChunked) {
                if (depth_stages <= 4) return small;
                if (image_mib < 256) return c_mib < (!shallow ? (image_mib < 100 ? 256 : 0) : image_mib < 30 ? 384 : image_mib < 100 ? 320 : 200) ? small : past(3);
                if (shallow && c_mib < 384) return small;
                if (!(needs_shift<T>(args) || (T::kSrcChunk == 16 && args.k_src_bytes % (2 * kStageChunks * T::kSrcChunk) != 0))) return 2;
                if (shallow) return args.m > 128 && args.m <= 192 ? small : Choice(3); // (three tiles of 64, but four of them in tiles of 128)
                return args.m > 1000 ? past(3) : Choice(3);
            }
            if (depth_stages <= 2) return c_mib < 384 ? small : halves && !bits ? past(3) : Choice(3);
            if (bits) { // (operands of an eighth)
                if (depth_stages <= 4) return c_mib < 320 ? small : Choice(args.m <= 160 || (args.m < 800 && c_mib > 640) ? 2 : 3);
                if (shallow) return c_mib < 384 ? small : Choice(args.m < 600 || c_mib > 1200 || (c_mib > 640 && args.m <= 1500) ? 2 : 3);
                if ((rows_at & 15) == 0) return halves || c_mib >= 300 ? past(3) : Choice(3);
                return c_mib < 512 ? small : Choice(3);
            }
            if (depth_stages <= 4) return c_mib < 320 ? small : halves ? past(3) : Choice(image_mib < 30 || args.m <= 128 ? 3 : 2);
            if (shallow) {
                int const wide = args.m <= 400 || T::kUnsigned || (args.m < 1024 && ((args.m + 127) / 128) % 2 != 0) ? 2 : best;
                if (c_mib < (image_mib < 10 ? 320 : 256)) return small;
                if (image_mib >= 256) return wide;
                if (c_mib < 320) return 3;
                return (rows_at & 7) == 0 ? past(3) : Choice(T::kUnsigned && image_mib < 100 ? 3 : wide);
            }
            if (image_mib < 256) return image_mib < 30 && c_mib < 240 ? Choice(3) : past(3);
            return args.m <= 400 || (T::kUnsigned && c_mib < 640) ? 2 : best;
        }
        return best;
    };
    // A in registers (see dots_resident_kernel) wherever there is such a kernel, C is most of the traffic and a strip is long enough for
    // what its start costs. Against the choice without it, rounds of three sets of operands and results, at 14,000 random shapes of all types
    // that it takes, 65 to 300,000 rows, C of 64 MiB to 2.4 GiB, the time is 0.81 in the mean (dots, euclidean and angular alike), and more by 3 per
    // cent at 35, 38 and 61 in 1000, by 10 per cent at 8 (on another machine 26, 29, 36 and 6). Of the slower angular ones a fifth are floats of 4 and 6 stages on
    // lines with images of 64 MiB and more and 257 to 2048 rows (0.96 in the mean of 109). At 4400 more shapes, where the lines lie: C under 64 MiB 0.98 to 1.05, strips
    // of fewer than 12 tiles 0.98 to 1.1 (of 12 to 15 up to 1.16), up to 64 rows 1.0. The angular finaliser is too much for few wavefronts (f16
    // 69 x 2,664,123 x 602 1.55, u4 318 x 137,089 x 1072 1.29).
    // Two blocks of rows, which ask half as often for the image, where that does not stay in the last-level cache beside C, and of more
    // rows the deeper the product (7400 shapes, each both ways): of 2 stages 1.03 of the time with one up to 8 MiB of image, 1.02 to 32, 1.01 to 64, then 0.93,
    // 0.87 from 80 to 256 MiB; of 4 stages 1.02 to 64 MiB, then 0.91, 0.88 to 112; of 6 stages 1.05 to 64 MiB, 1.02 to 80, then 0.90. From there on
    // by workgroups of 256 rows: two 0.90 (2 stages), 1.01 (4) and 1.05 (6), three 0.87, 0.94 and 1.01, four 0.85, 0.86 and 0.99, five 0.88, 0.80 and 0.91. (i8
    // 1024 x 1,048,576 x 768 1195 us and 1080.)
    // Left out: short dots whose strips write in step (see ResidentPlan) with more than eight workgroups of rows (i8 31,126 x 2048 x 256 77 us, 52
    // through tiles; without A in registers 0.87 of the time in the mean of 471 calls of two stages, 0.92 of 381 of four, but of e2m3 and
    // u8, whose tiles widen or sum A, 1.13 and 1.07 at four), and floats of 8 stages off the lines with up to 128 rows (0.97 of 415).
    auto resident_blocks = [&](GemmArgs const &args) -> int {
        if (triangle || args.m <= 64 || (uint64_t)args.m * args.n * 4 < (64ull << 20) || !resident_kernel<T>(args, 1)) return 0;
        ResidentPlan const plan = resident_plan(args.m, args.n_tiles, 32, args.c_stride);
        uint32_t const stages = args.k_chunks / kStageChunks;
        bool const lines = (((uintptr_t)args.c | args.c_stride) & 127) == 0;
        uint64_t const image_mib = ((uint64_t)args.n_tiles * args.k_chunks * kTileChunkBytes) >> 20;
        if (plan.strip_tiles < 16 || (args.metric == 1 && plan.waves < 6)) return 0;
        bool const two = image_mib >= (stages <= 4 ? 64 : 80) && args.m > (stages <= 2 ? 256 : stages <= 4 ? 512 : 768) && resident_kernel<T>(args, 2);
        if (args.metric == 0 && stages <= (T::kDtype == kE2M3 || T::kUnsigned ? 2 : 4) && plan.in_step && plan.blocks > 8 && !two) return 0;
        if (args.metric == 0 && T::kChunked && stages == 8 && args.m <= 128 && !lines) return 0;
        return two ? 2 : 1;
    };
    if (config == 8 || config == 9) {
        if (!triangle && resident_kernel<T>(g, config - 7)) return launch_resident<T>(g, stream, config - 7, planned);
        config = 4;
    }
    if (chosen_here)
        if (int const blocks = resident_blocks(g)) {
            hipError_t const status = launch_resident<T>(g, stream, blocks, planned);
            if (!planned) return status;
        }
    Choice const chosen = chosen_here ? choose(g, 1) : Choice(config);
    config = chosen.config, g.store_policy = chosen.store_policy;
    if (config == 7) {
        if constexpr (!T::kDeepOnly)
            if (!triangle && strips_possible<T>(g)) return launch_strips<T>(g, stream, planned);
        config = 4;
    }
    if ((T::kChunked || needs_shift<T>(g)) && (config == 1 || config == 5)) config = 2;
    if (triangle && config >= kTriangleConfigs) config = 4;
    auto grid_of = [](GemmArgs const &args, int c, TriangleScratch const &scratch) {
        uint32_t const bm = kConfigs[c].tm * 32, bn = kConfigs[c].tn * 128;
        TriangleGrid grid;
        grid.tiles_m = (args.m + bm - 1) / bm, grid.tiles_n = (args.n + bn - 1) / bn;
        grid.bm_log2 = log2_of(bm), grid.bn_log2 = log2_of(bn), grid.shift = args.tri_shift;
        grid.bands = (grid.tiles_m + kTileBand - 1) / kTileBand, grid.list = scratch.words;
        return grid;
    };

    // A triangular grid rarely fills a whole number of rounds of the persistent workgroups, and a last round that
    // is mostly empty costs as much as a full one. When that last round would be less than half full, the tile rows
    // from the top that fill whole rounds go to this tile shape and the rows below them, the narrow end of the
    // triangle, to a second launch with small tiles that spreads them over the whole device. (Not 128 x 128 with A out of the
    // image, two workgroups per compute unit: i8 8192 x 768 68 us in two launches, 63 in one; bf16 96 and 91.)
    if (triangle && (chosen_here || (forced & 0x80)) && config < 4 && !(config == 3 && triangle->self && chosen_here)) {
        int slots = 0;
        GemmArgs probe = g;
        hipError_t e = launch_config<T>(probe, stream, triangle, config, &slots);
        if (e != hipSuccess) return e;
        uint64_t const live = tiles_of(g, config);
        uint64_t const rounds = slots > 0 ? live / (uint64_t)slots : 0, rest = slots > 0 ? live % (uint64_t)slots : 0;
        if (rounds >= 1 && rest > 0 && rest * 2 <= (uint64_t)slots) {
            uint32_t const bm = kConfigs[config].tm * 32, bn = kConfigs[config].tn * 128;
            uint32_t const tiles_m = (g.m + bm - 1) / bm, tiles_n = (g.n + bn - 1) / bn;
            uint64_t count = 0;
            uint32_t keep = 0; // tile rows that stay with the large tiles
            for (; keep < tiles_m; ++keep) {
                uint32_t const from = first_live_tile(keep, log2_of(bm), log2_of(bn), g.tri_shift);
                uint64_t const here = from < tiles_n ? tiles_n - from : 0;
                if (count + here > rounds * (uint64_t)slots) break;
                count += here;
            }
            if (keep > 0 && keep < tiles_m) {
                GemmArgs top = g, bottom = g;
                top.m = keep * bm;
                bottom.m = g.m - top.m;
                bottom.a += (uint64_t)top.m * g.a_stride, bottom.c += (uint64_t)top.m * g.c_stride;
                bottom.tri_shift = g.tri_shift + top.m;
                // each launch builds its tile list in its own half of the scratch memory
                size_t const half = triangle->bytes / 2 / 8 * 8;
                TriangleScratch const first_half = {triangle->words, half, nullptr, triangle->self}, second_half = {triangle->words + half / 4, half, nullptr, triangle->self};
                int const narrow = choose(bottom, config + 1).config;
                if (triangle->plan) {
                    triangle->plan->grid[0] = grid_of(top, config, first_half), triangle->plan->grid[1] = grid_of(bottom, narrow, second_half);
                    return hipSuccess;
                }
                if ((e = launch_config<T>(top, stream, &first_half, config)) != hipSuccess) return e;
                return launch_config<T>(bottom, stream, &second_half, narrow);
            }
        }
    }
    if (triangle && triangle->plan) {
        triangle->plan->grid[0] = grid_of(g, config, *triangle), triangle->plan->grid[1] = TriangleGrid {};
        return hipSuccess;
    }
    if (planned) {
        planned->shape = (uint32_t)config, planned->store_policy = g.store_policy, planned->units = (uint32_t)tiles_of(g, config);
        planned->direct = config == 1 ? goes_direct<T, 8, 2>(g) : config == 2 ? goes_direct<T, 4, 2>(g) : config == 3 && goes_direct<T, 4, 1>(g);
        return hipSuccess;
    }
    return launch_config<T>(g, stream, triangle, config);
}

inline int widest_load(void const *p, size_t stride) {
    uintptr_t const bits = (uintptr_t)p | (uintptr_t)stride;
    if (!(bits & 15)) return 16;
    if (!(bits & 7)) return 8;
    if (!(bits & 3)) return 4;
    if (!(bits & 1)) return 2;
    return 1;
}

#pragma endregion Packed product

} // namespace

#endif // NUMKONG_AMD_DOTS_GFX950_HPP
