// Q8_K activation quantizer for gfx950: one wave per 256-value block, 4 values per lane
// (block quantization in q8k_block.h).
#include "kq_device.h"
#include "kq_internal.h"
#include "q8k_block.h"

namespace kq {

__global__ void __launch_bounds__(256)
k_q8k_quantize(const float* __restrict__ x, int64_t ldx, int G, int nblocks, uint8_t* __restrict__ xq) {
    // every argument load issued before the first wait (one round trip to the arguments, not two)
    const int nthr = blockDim.x;
    KQ_ARGS_READY("s"(x), "s"(ldx), "s"(G), "s"(nblocks), "s"(xq), "s"(nthr));
    const int lane = threadIdx.x & 63;
    const int blk = blockIdx.x * (nthr >> 6) + (threadIdx.x >> 6);
    if (blk >= nblocks) return;
    const int n = blk / G, g = blk - n * G;
    const f32x4 v = *reinterpret_cast<const f32x4_a4*>(x + (int64_t)n * ldx + (int64_t)g * QK + 4 * lane);
    const float e[4] = {v.x, v.y, v.z, v.w};
    q8k_block_store(e, lane, xq + (int64_t)blk * Q8K_BYTES);
}

// The same, also writing the quants in the prefill GEMM's fragment order (gemm_q8k.hip: xf[m/32][g][ks][l][16 B]
// = qs bytes 32ks + 16(l/32) .. +15 of row 32(m/32) + l%32).  A workgroup takes one super-block of QF_ROWS consecutive
// rows, a wave each; their quants meet in LDS, so that the 16-byte pieces of consecutive rows leave as whole 128-byte
// lines (written from each wave's own registers, 4 bytes a lane, every line was written in 32 parts).
// Rows M .. Mpad-1 are zero in the fragment copy and absent from the Q8_K rows, as in the stand-alone fragment copy.
// 2048 rows of 4096 / 12288 15.0 / 36.8 -> 12.9 / 31.6 us, 256 rows of 12288 7.6 -> 6.6 us; bound by memory there.
constexpr int QF_ROWS = 8;
__global__ void __launch_bounds__(64 * QF_ROWS)
k_q8k_quantize_frag(const float* __restrict__ x, int64_t ldx, int G, int M, uint8_t* __restrict__ xq,
                    uint8_t* __restrict__ xf) {
    __shared__ __attribute__((aligned(16))) uint32_t qs[QF_ROWS][64 + 4];
    KQ_ARGS_READY("s"(x), "s"(ldx), "s"(G), "s"(M), "s"(xq), "s"(xf));
    const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
    const int rg = blockIdx.x / G, g = blockIdx.x - rg * G, n0 = rg * QF_ROWS, n = n0 + row;
    uint32_t q = 0u;
    if (n < M) {
        const f32x4 v = *reinterpret_cast<const f32x4_a4*>(x + (int64_t)n * ldx + (int64_t)g * QK + 4 * lane);
        const float e[4] = {v.x, v.y, v.z, v.w};
        q = q8k_block_store(e, lane, xq + ((int64_t)n * G + g) * Q8K_BYTES);
    }
    qs[row][lane] = q;
    __syncthreads();
    if (threadIdx.x < 16 * QF_ROWS) {       // piece c = 2 ks + half of row r
        const int c = threadIdx.x / QF_ROWS, r = threadIdx.x % QF_ROWS;
        uint8_t* const fo = xf + (((int64_t)(n0 >> 5) * G + g) * 8 + (c >> 1)) * 1024 + ((n0 & 31) + r + 32 * (c & 1)) * 16;
        *reinterpret_cast<u32x4*>(fo) = *reinterpret_cast<const u32x4*>(&qs[r][4 * c]);
    }
}

void launch_q8k_quantize_frag(const float* x, int64_t ldx, int C, int M, int Mpad, uint8_t* xq, uint8_t* xf,
                              hipStream_t s) {
    const int G = C / QK;
    hipLaunchKernelGGL(k_q8k_quantize_frag, dim3(Mpad / QF_ROWS * G), dim3(64 * QF_ROWS), 0, s, x, ldx, G, M, xq, xf);
}

void launch_q8k_quantize(const float* x, int64_t ldx, int C, int N, uint8_t* xq, hipStream_t s) {
    const int G = C / QK;
    const int nblocks = N * G;
    const int wpb = 4;
    dim3 grid((nblocks + wpb - 1) / wpb), block(64 * wpb);
    hipLaunchKernelGGL(k_q8k_quantize, grid, block, 0, s, x, ldx, G, nblocks, xq);
}

}  // namespace kq
