// Slot lists of the flash-EMA attention: for every 32-step block, the valid slots whose
// counters can be nonzero at one of its steps.
//
// A slot contributes to a block only if its chunk-start state is nonzero or its token occurs
// in the match window before the block's last step: otherwise its counters are zero at all 32
// steps, its gate SiLU(0) = 0, its score and value 0 and every gradient term 0 (dW_pe's too,
// whose other factor is the counter).  Such a slot only adds e^0 to the softmax sum, which the
// forward adds as a count.  Tokens that the history does not hold stay out of the blocks before
// their first occurrence: 20 % of the (step, slot) pairs at B16 T4096 with a 4096-token
// history, 4 % at B56 T512, about 40 % of a chunk without a history.  The lists keep the
// slots' order, so the sums run over the remaining terms in the same order.  Measured: B16 T4096
// N128 backward 107.1 -> 83.7 ms and forward 38.5 -> 33.0 ms; B56 T512 N64 21.6 -> 20.1 and
// 10.8 -> 10.7 ms; a forward over one 10 001-step sequence 7.78 -> 5.31 ms.
//
// Bound: the read of C_bounds in rows of N floats by whole waves.  Per slot and chunk of 64 steps
// 4 N bytes and 8 of the id are read and up to 32 written (two entries): the rest is a sixth of
// the rows at N = 64, a twelfth at 128 and over half at 16.  B56 T512 N64 216 MB in 70 us, B16
// T4096 N128 1.36 GB in 454 us (3.0 TB/s both); a grid of few (sequence, chunk) pairs is bound by
// the latency of a workgroup's rounds of 512 slots instead (B8 T512, 64 workgroups: 41 us).
#include "flash_common.h"

namespace mb {

constexpr int kListThreads = 512;

struct ListArgs {
    const int64_t* x;
    int64_t x_sb, x_sl;
    const int64_t* unique;
    const float* Cb;
    int B, L, K, N, Np, Br, nc, ntb;
    BatchMeta* list;
    SlotCount* count;
    int32_t* order;
};

// Byte offsets of the counts and of the order behind the lists' entries.
static int64_t slot_count_offset(int64_t blocks, int K) { return blocks * K * (int64_t)sizeof(BatchMeta); }
static int64_t slot_order_offset(int64_t blocks, int K) {
    return slot_count_offset(blocks, K) + blocks * (int64_t)sizeof(SlotCount);
}

// One workgroup per (sequence, chunk start): with Br = 64 a chunk's two blocks share the states
// and the window, otherwise each block has its own.  Each wave takes 64 slots per round.
// VEC: rows are read as float4 (Np % 4 == 0).
template <bool VEC>
__global__ void __launch_bounds__(kListThreads)
flash_slot_list_kernel(ListArgs a) {
    constexpr int NW = kListThreads / 64;
    __shared__ int64_t win[kMaxWin];
    __shared__ int wsum[2][NW];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int per = a.Br == 64 ? 2 : 1;  // blocks per workgroup
    const int groups = (a.ntb + per - 1) / per;
    const int b = blockIdx.x / groups;
    const int blk0 = (blockIdx.x % groups) * per;
    const int cbi = blk0 * kTB / a.Br;
    const int cb = cbi * a.Br;
    if (threadIdx.x < kMaxWin) {
        const int pos = cb + threadIdx.x;
        win[threadIdx.x] = pos < a.L ? a.x[(int64_t)b * a.x_sb + (int64_t)pos * a.x_sl] : (int64_t)-1;
    }
    __syncthreads();
    const float* rows = a.Cb + ((int64_t)b * a.nc + cbi) * a.K * a.Np;
    const int lpr = VEC ? (a.N <= 32 ? 8 : a.N <= 64 ? 16 : 32) : 64;  // lanes per row
    const int rpi = 64 / lpr;                                          // rows per load
    int run[2] = {0, 0}, nvalid = 0;
    for (int k0 = 0; k0 < a.K; k0 += kListThreads) {
        const int kw = k0 + 64 * wave;
        const int k = kw + lane;
        const int64_t u = k < a.K ? a.unique[(int64_t)b * a.K + k] : (int64_t)-1;
        // bit l of the lane's slot: any rate of its state nonzero (NaN counts as nonzero)
        bool state = false;
        if (kw < a.K) {  // (uniform across the wave)
#pragma unroll 8
            for (int it = 0; it < lpr; ++it) {
                const int r = kw + it * rpi + lane / lpr;
                const int n = (lane % lpr) * (VEC ? 4 : 1);
                bool nz = false;
                if (r < a.K) {
                    const float* p = rows + (int64_t)r * a.Np;
                    if (VEC) {
                        if (n < a.N) {
                            const float4 v = *reinterpret_cast<const float4*>(p + n);
                            nz = v.x != 0.f || (n + 1 < a.N && v.y != 0.f) || (n + 2 < a.N && v.z != 0.f) ||
                                 (n + 3 < a.N && v.w != 0.f);
                        }
                    } else {
                        nz = (n < a.N && p[n] != 0.f) || (n + 64 < a.N && p[n + 64] != 0.f);
                    }
                }
                const uint64_t m = __ballot(nz) >> (lane % rpi * lpr % 64);
                if (it == lane / rpi) state = (VEC ? m & ((1ull << (lpr & 63)) - 1ull) : m) != 0;
            }
        }
        uint64_t mask = 0;
        for (int p = 0; p < kMaxWin; ++p) mask |= (uint64_t)(win[p] == u) << p;
        uint64_t act[2];
        for (int j = 0; j < per; ++j) {
            // occurrences before the block's last step gate a step of it
            const int end = (blk0 + j) * kTB - cb + kTB - 1;
            const bool in = (blk0 + j) < a.ntb && u >= 0 && (state || (mask & ((1ull << end) - 1ull)));
            act[j] = __ballot(in);
            if (lane == 0) wsum[j][wave] = __popcll(act[j]);
        }
        nvalid += __popcll(__ballot(u >= 0));
        __syncthreads();
        for (int j = 0; j < per; ++j) {
            int before = run[j], total = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w < wave) before += wsum[j][w];
                total += wsum[j][w];
            }
            if ((act[j] >> lane) & 1) {
                const int at = before + __popcll(act[j] & ((1ull << lane) - 1ull));
                a.list[((int64_t)b * a.ntb + blk0 + j) * a.K + at] = BatchMeta{mask, slot_row(u), k};
            }
            run[j] += total;
        }
        __syncthreads();
    }
    if (lane == 0) wsum[0][wave] = nvalid;
    __syncthreads();
    if (threadIdx.x < per && blk0 + (int)threadIdx.x < a.ntb) {
        int valid = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) valid += wsum[0][w];
        a.count[(int64_t)b * a.ntb + blk0 + threadIdx.x] = SlotCount{threadIdx.x ? run[1] : run[0], valid};
    }
}

// The blocks by the length of their lists, longest first: the attention's workgroups run in this
// order, so that lists of very different lengths (documents' chunks) still end together.  A
// counting sort over 1024 lengths; equal ones come in any order.  One workgroup, 5 us.
__global__ void __launch_bounds__(1024)
flash_slot_order_kernel(const SlotCount* __restrict__ count, int blocks, int K, int32_t* __restrict__ order) {
    constexpr int BINS = 1024;
    __shared__ int bins[BINS];
    __shared__ int scratch[64];
    bins[threadIdx.x] = 0;
    __syncthreads();
    auto bin = [&](int i) { return BINS - 1 - (int)((int64_t)count[i].active * (BINS - 1) / K); };  // 0: longest
    for (int i = threadIdx.x; i < blocks; i += blockDim.x) atomicAdd(&bins[bin(i)], 1);
    __syncthreads();
    int total;
    const int mine = bins[threadIdx.x];
    const int start = block_exclusive_scan(mine, scratch, total);
    bins[threadIdx.x] = start;
    __syncthreads();
    for (int i = threadIdx.x; i < blocks; i += blockDim.x) order[atomicAdd(&bins[bin(i)], 1)] = i;
}

int flash_validate(const char* who, const FlashArgs& a, int hd);

// Sets a call's list pointers (NULL: the call walks every slot).
void flash_use_lists(FlashArgs& a, const void* lists) {
    if (!lists || a.B == 0 || a.L == 0 || a.K == 0) return;
    const int64_t blocks = (int64_t)a.B * ((a.L + kTB - 1) / kTB);
    a.list = static_cast<const BatchMeta*>(lists);
    const char* base = static_cast<const char*>(lists);
    a.nlist = reinterpret_cast<const SlotCount*>(base + slot_count_offset(blocks, a.K));
    a.order = reinterpret_cast<const int32_t*>(base + slot_order_offset(blocks, a.K));
}

}  // namespace mb

using namespace mb;

extern "C" int64_t mb_flash_ema_slot_lists_bytes(int B, int L, int K) {
    if (B <= 0 || L <= 0 || K <= 0) return 0;
    const int64_t blocks = (int64_t)B * ((L + kTB - 1) / kTB);
    return slot_order_offset(blocks, K) + blocks * (int64_t)sizeof(int32_t);
}

extern "C" int mb_flash_ema_slot_lists(const int64_t* x, int64_t x_sb, int64_t x_sl, const int64_t* unique,
                                       const float* C_bounds, int B, int L, int K, int N, int Np, int nc, int Br,
                                       void* slot_lists, void* stream) {
    FlashArgs f{};
    f.B = B; f.H = 1; f.L = L; f.K = K; f.N = N; f.Np = Np; f.Br = Br; f.nc = nc;
    int rc = flash_validate("mb_flash_ema_slot_lists", f, 64);
    if (rc) return rc;
    if (B == 0 || L == 0 || K == 0) return MB_OK;
    MB_REQUIRE(x && unique && C_bounds && slot_lists, "mb_flash_ema_slot_lists: null pointer");
    MB_REQUIRE(((uintptr_t)slot_lists & 15) == 0, "mb_flash_ema_slot_lists: slot_lists must be 16-byte aligned");
    ListArgs a{};
    a.x = x; a.x_sb = x_sb; a.x_sl = x_sl; a.unique = unique; a.Cb = C_bounds;
    a.B = B; a.L = L; a.K = K; a.N = N; a.Np = Np; a.Br = Br; a.nc = nc;
    a.ntb = (L + kTB - 1) / kTB;
    f.list = nullptr;
    flash_use_lists(f, slot_lists);
    a.list = const_cast<BatchMeta*>(f.list);
    a.count = const_cast<SlotCount*>(f.nlist);
    a.order = const_cast<int32_t*>(f.order);
    const int per = Br == 64 ? 2 : 1;
    const int64_t grid = (int64_t)B * ((a.ntb + per - 1) / per);
    MB_REQUIRE((int64_t)B * a.ntb <= INT32_MAX, "mb_flash_ema_slot_lists: B=%d, L=%d too large", B, L);
    // float4 rows need 16-byte rows
    if (Np % 4 == 0 && ((uintptr_t)C_bounds & 15) == 0)
        hipLaunchKernelGGL(flash_slot_list_kernel<true>, dim3((unsigned)grid), dim3(kListThreads), 0,
                           (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL(flash_slot_list_kernel<false>, dim3((unsigned)grid), dim3(kListThreads), 0,
                           (hipStream_t)stream, a);
    hipLaunchKernelGGL(flash_slot_order_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, a.count, B * a.ntb, K,
                       a.order);
    return check_launch("mb_flash_ema_slot_lists");
}
