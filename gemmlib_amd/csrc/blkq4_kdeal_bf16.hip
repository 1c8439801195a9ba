// The tile kernel whose waves are dealt whole k tiles for bf16 activations, scales and outputs: the same source as for fp16,
// with the element type switched (conversion of the weights, MFMA instruction, rounding of the outputs, bias).
#define BLKQ4_KDEAL_BF16 1
#include "blkq4_kdeal.hip"
