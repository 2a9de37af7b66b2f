// paged_decode_row.hip - the matrix-core decode of a small batch in one launch: a workgroup per row and KV head.
//
// The split decode (paged_decode_mfma.hip) deals the pages of all rows evenly over the chip and folds the pieces of
// each row with a second kernel.  That pays once there is enough to stream; a small batch of short rows pays more for the
// second launch, the partials and the search for its rows than for its pages.  Here a workgroup of eight waves takes one
// row and one KV head (or block of 16 of its query heads): its waves stream shares of the row's pages with the same code
// (decode_wg with ROW), meet in LDS and write the output.
#define FFKV_DEVICE_BODIES_ONLY 1
#include "paged_decode_mfma.hip"
#undef FFKV_DEVICE_BODIES_ONLY

namespace ffkv
{

namespace
{

constexpr int kRowWaves = 8;  // waves per workgroup: two per SIMD, as the registers of most variants allow

// LDS of a workgroup whose blocks have up to `heads` query heads: the waves' V tiles, and over them the waves'
// accumulators and (max, denominator) pairs once all pages are done.
template <int D>
constexpr int row_lds_bytes(int heads)
{
    const int v = kRowWaves * kBlockSize * D * 2;
    const int state = kRowWaves * heads * D * 4 + kRowWaves * 16 * 8;
    return v > state ? v : state;
}
static_assert(row_lds_bytes<256>(16) <= 160 * 1024, "a workgroup's LDS fits a CU");

template <int CT, int QT, int D>
__global__ __launch_bounds__(64 * kRowWaves) __attribute__((amdgpu_waves_per_eu(2, 8)))
void paged_decode_row(DecodeArgs a)
{
    extern __shared__ __align__(16) uint8_t s_row[];
    decode_wg<CT, QT, D, false, true>(a, static_cast<int>(blockIdx.y), static_cast<int>(blockIdx.x), 0, kRowWaves,
                                      reinterpret_cast<uint16_t*>(s_row));
}

template <int CT, int QT, int D>
hipError_t launch_row3(const DecodeArgs& a, hipStream_t stream)
{
    const int  hb = (a.group + 15) / 16;
    const int  lds = row_lds_bytes<D>(a.group < 16 ? a.group : 16);
    const dim3 grid(static_cast<unsigned>(a.num_kv_heads * hb), static_cast<unsigned>(a.batch));
    hipLaunchKernelGGL((paged_decode_row<CT, QT, D>), grid, dim3(64 * kRowWaves), static_cast<unsigned>(lds), stream, a);
    return hipGetLastError();
}

template <int CT, int QT>
hipError_t launch_row2(const DecodeArgs& a, hipStream_t stream)
{
    switch (a.head_dim)
    {
        case 64:
            return launch_row3<CT, QT, 64>(a, stream);
        case 80:
            return launch_row3<CT, QT, 80>(a, stream);
        case 96:
            return launch_row3<CT, QT, 96>(a, stream);
        case 112:
            return launch_row3<CT, QT, 112>(a, stream);
        case 128:
            return launch_row3<CT, QT, 128>(a, stream);
        default:
            return launch_row3<CT, QT, 256>(a, stream);
    }
}

template <int CT>
hipError_t launch_row1(const DecodeArgs& a, hipStream_t stream)
{
    switch (a.qo_dtype)
    {
        case F32:
            return launch_row2<CT, F32>(a, stream);
        case F16:
            return launch_row2<CT, F16>(a, stream);
        default:
            return launch_row2<CT, BF16>(a, stream);
    }
}

}  // namespace

// One CU draws about 47 GB/s of pages whatever its waves keep in flight (8 or 12 waves, two or three pages each, measured
// alike), so a workgroup takes 6 us and 11 us per 512 KiB of its row; the split decode takes 9 to 12 us for the smallest
// batches and 13 to 27 us from 16 rows on.  The row's length is not known here, only its bound (max_context_len or the
// table's width), so the rule holds for rows as long as that.  Whole calls (append included), split -> row, us:
//   up to 256 KiB of K and V per (row, KV head), up to 512 workgroups: 4 rows of 17 to 255 tokens at 16/8 heads 9.3 -> 6.9;
//   at 32/8 heads 1 row of 500 tokens 9.7 -> 9.2, 8 rows of 100 to 500 10.5 -> 9.4, 16 rows 13.3 -> 9.8, 64 rows 23.1 ->
//   21.3; 32 rows of 500 to 1000 tokens of 64 dims 17.6 -> 11.6, on int8 pages of 128 dims 25.9 -> 21.4
//   up to 512 KiB, 128 to 256 workgroups: 16 rows of 500 to 1000 tokens 16.8 -> 16.1, 32 rows 25.2 -> 21.1, 32 rows of 200
//   to 400 tokens of 256 dims 27.3 -> 19.6
// Beyond that the split is ahead: 1 row of 1000 tokens 10.6 against 13.4, 8 rows of 200 to 800 11.7 against 12.9, 48 rows of
// 100 to 1000 26.9 against 27.3 (more workgroups than CUs), 128 rows of 50 to 250 24.3 against 26.5.
bool decode_use_row(const DecodeArgs& a)
{
    const int64_t wgs = static_cast<int64_t>(a.batch) * a.num_kv_heads * ((a.group + 15) / 16);
    const int64_t es = a.cache_dtype == I8 || a.cache_dtype == FP8 ? 1 : 2;
    const int64_t bytes = 2 * es * a.head_dim * a.cap_tokens;  // K and V of a row and KV head, at most
    if (bytes <= (256 << 10)) return wgs <= 512;
    return bytes <= (512 << 10) && wgs >= 128 && wgs <= 256;
}

hipError_t launch_decode_row(const DecodeArgs& a, hipStream_t stream)
{
    switch (a.cache_dtype)
    {
        case BF16:
            return launch_row1<BF16>(a, stream);
        case F16:
            return launch_row1<F16>(a, stream);
        case I8:
            return launch_row1<I8>(a, stream);
        default:
            return launch_row1<FP8>(a, stream);
    }
}

}  // namespace ffkv
