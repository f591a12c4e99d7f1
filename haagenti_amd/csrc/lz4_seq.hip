// Batched raw-LZ4 block decoder: one wavefront per block, sequences parsed
// in batches and copied lane-parallel (the decoder is in lz4_seq.hpp).
#include <type_traits>

#include "lz4_seq.hpp"

namespace hh {
namespace {

template <uint32_t R, uint32_t S, class PART>
__global__ __launch_bounds__(64) void lz4_seq_kernel(Lz4Batch B, PART part) {
    using D = seq::SeqDec<R, S, false>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x;
    if (blockIdx.x >= B.nblocks) return;
    uint32_t b = blockIdx.x + B.first;
    b = b >= B.nblocks ? b - B.nblocks : b;

    int32_t code = HH_OK, detail = HH_CORRUPT_NONE;
    uint64_t pos = 0, req = 0;

    const uint64_t ioff = B.in_off[b];
    const uint32_t ilen = B.in_len[b];
    const uint64_t oofs = B.out_off[b];
    const uint32_t ocap = B.out_cap[b];
    if (!part.takes(B.out + oofs, ocap)) return;
    // beside other kernels (a split layer) the chain issues before them:
    // 217 against 265 us for a Llama-3-8B layer's tensors of retention 0.10
    // and 0.20 (190 with the device to itself)
    if constexpr (std::is_same_v<PART, Lz4Some<true>>) __builtin_amdgcn_s_setprio(3);
    const bool out_ok = oofs <= B.out_total && (uint64_t)ocap <= B.out_total - oofs;
    uint8_t *out = B.out + oofs;
    D d;
    seq::lds8 *lds = (seq::lds8 *)smem;
    d.ring = lds;
    d.tab = reinterpret_cast<seq::lds32 *>(lds + R);
    d.stage = lds + R + D::kTabLds + D::kSFront;
    d.gbuf = B.in;
    d.gsz = B.in_total;
    d.ioff = ioff;
    d.a0 = (uint32_t)((uintptr_t)out & 15u);
    d.obase = out - d.a0;
    d.cap = ocap;
    d.sb = 0;
    d.at_end = false;
    d.op = 0;
    d.fl = 0;
    d.lane = lane;

    if (ioff > B.in_total || (uint64_t)ilen > B.in_total - ioff || !out_ok) {
        code = HH_ERR_INVALID_ARGUMENT;
    } else {
        seq::decode_block(d, ilen, code, detail, pos, req);
        if (code == HH_OK) d.flush(true);
    }
    // a failed block's output reads as zeros (the reference returns no output)
    if (code != HH_OK && out_ok) {
        __asm__ __volatile__("" ::: "memory");
        wave_zero_fill(out, d.cap, lane);
    } else if (code == HH_OK && B.zero_tail && d.op < d.cap) {
        wave_zero_fill(out + d.op, d.cap - d.op, lane);
    }
    if (lane == 0) {
        hh_block_status st;
        st.code = code;
        st.detail = detail;
        st.position = pos;
        st.required = req;
        st.written = code == HH_OK ? d.op : 0;
        B.status[b] = st;
    }
}

template <uint32_t R, uint32_t S, class PART = Lz4All>
hipError_t launch_seq(const Lz4Batch &B, hipStream_t s, const PART &part = PART{}) {
    constexpr uint32_t lds = seq::SeqDec<R, S, false>::kLds;
    hipError_t e = hipFuncSetAttribute((const void *)lz4_seq_kernel<R, S, PART>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((lz4_seq_kernel<R, S, PART>), dim3(B.nblocks), dim3(64), lds, s, B, part);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_lz4_seq(const Lz4Batch &B, uint32_t ring_kib, hipStream_t s) {
    if (B.nblocks == 0) return hipSuccess;
    switch (ring_kib) {
        case 8: return launch_seq<8192, 2048>(B, s);
        default: return launch_seq<4096, 4096>(B, s);
    }
}

hipError_t launch_lz4_seq_in(const Lz4Batch &B, const Lz4Ranges &r, hipStream_t s) {
    if (B.nblocks == 0) return hipSuccess;
    return launch_seq<4096, 4096>(B, s, Lz4Some<true>{r});
}

}  // namespace hh
