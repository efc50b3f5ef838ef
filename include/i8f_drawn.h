/*
 * An entry point that follows the random number generator of one version of torch, kept apart from the ABI of i8f.h for that
 * reason: a caller under another version draws the noise itself and calls i8f_lora_merge_sr.
 */
#ifndef I8F_DRAWN_H
#define I8F_DRAWN_H

#include "i8f.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * The low-rank form of i8f_lora_merge_sr for one LoRA or a stack of them, on noise that is drawn here: noise[n,k] is element
 * e = n K + k of what torch.rand (torch 2.10 on ROCm) writes on this GPU from a generator seeded with `seed`, whose launch has
 * `lanes` threads (256 to a block; min(ceil(N K / 256), blocks that the GPU holds at once) blocks).  With i = e / lanes and x
 * the word i % 4 of Philox 4x32-10 (key: seed; counter: (i / 4, 0, e % lanes, 0)), it is RN(RN(x) 2^-32 + 2^-32), and 0 where
 * that is 1.  A stack (count > 1) is one product of the factors side by side, in order, each `down` times its `mult`
 * (rounded); of one LoRA mult is not looked at.  The result is that of i8f_lora_merge_sr on these factors and this noise, bit
 * for bit (INT8LoRAPatchAdapter / INT8MergedLoRAPatchAdapter.calculate_weight, int8_quant.py:293-318, 382-404).
 * up [N,rank] and down [rank,K] of each are float.  At most 8 LoRAs, K % 16 == 0, K < 2^24, the sum of the ranks a
 * multiple of 4 and <= 256, N K <= 2^29, lanes % 256 == 0, lanes <= 2^24, N K / (4 lanes) within the 65535 blocks of a
 * launch, a stack's (N + K) rank < 2^31, w, w_out, workspace and the `up` of a
 * single LoRA 16-byte aligned; else I8F_ERR_UNSUPPORTED.  workspace: any contents.  w_out may equal w.
 */
typedef struct {
    const float *up, *down;
    int64_t rank;
    float mult;
} i8f_lora_factors;
int64_t i8f_lora_merge_sr_drawn_workspace_bytes(int64_t N, int64_t K, int64_t rank, int count);
int i8f_lora_merge_sr_drawn(const int8_t *w, const float *w_scale, float w_scale_host, int scale_mode,
                            const i8f_lora_factors *factors, int count, float lora_scale,
                            uint64_t seed, int64_t lanes, int64_t N, int64_t K, int8_t *w_out,
                            void *workspace, int64_t workspace_bytes, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* I8F_DRAWN_H */
