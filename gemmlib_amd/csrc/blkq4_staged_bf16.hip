// The streaming kernel with rows staged slice by slice for bf16 activations, scales and outputs: the same source as for
// fp16, with the element type switched (conversion of the weights, MFMA instruction, rounding of the outputs, bias).
#define BLKQ4_STAGED_BF16 1
#include "blkq4_staged.hip"
