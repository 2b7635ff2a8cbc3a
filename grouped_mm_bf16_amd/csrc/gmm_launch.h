// Internal interface between the C ABI (gmm_api.hip) and the kernel families.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/grouped_mm_hip.h"
#include "gmm_sched.h"

// Each returns 0 on success, 1 if the launch failed, -1 if the dtype pair is unsupported.
// `kernel`: the one that was launched (gmm_kernel).
int gmm_launch_generic(GmmParams p, int in_dtype, int out_dtype, int num_cus, hipStream_t stream, int& kernel);

// Register-staged MFMA kernel for operands of any alignment (gmm_staged.hip): each operand contiguous along one of
// its dimensions.  Returns like gmm_launch_generic, the kernel is GMM_KERNEL_ANY.
bool gmm_staged_eligible(const GmmParams& p);
// Of the 16-bit products that the assembly tile could take: true for those that the register-staged kernel runs faster.
bool gmm_staged_preferred(const GmmParams& p, int num_cus);
// Those among them that are cut along K for it (needs a workspace).
bool gmm_staged_cut_preferred(const GmmParams& p, int num_cus);
// Of the products without alignment: true for those that the element-wise kernel runs faster.
bool gmm_element_preferred(const GmmParams& p, int in_dtype, int num_cus);
int gmm_launch_staged(GmmParams p, int in_dtype, int out_dtype, int num_cus, hipStream_t stream);
// Would this launch use a workspace of p.ws_parts slots?
bool gmm_staged_uses_workspace(const GmmParams& p, int in_dtype, int num_cus);

// Zeros in the rows (jagged rows) or columns (jagged columns) of the output that no group owns.
int gmm_launch_zero_unowned(const GmmParams& p, int out_dtype, hipStream_t stream);

// Operand layout facts the host derived from strides.
struct GmmLayout {
  bool a_kc;  // A contiguous along K (row-major); otherwise contiguous along M
  bool b_kc;  // B contiguous along K (column-major); otherwise contiguous along N
};

// Tile configurations of the MFMA family.
// REG: tiles staged through registers, compiler-scheduled (takes every aligned layout and the
//      jagged-column / unaligned jagged-contraction cases).
// ASM: generated assembly tile with direct-to-LDS copies (the fast one).
enum GmmMfmaConfig : int { GMM_CFG_REG_256x256 = 0, GMM_CFG_ASM_256x256 = 1, GMM_CFG_COUNT };

// bf16 inputs only; out_dtype bf16 or fp32.  Returns like gmm_launch_generic.
int gmm_launch_mfma(GmmParams p, GmmLayout lay, int in_dtype, int out_dtype, int config, int num_cus, hipStream_t stream);
bool gmm_mfma_uses_workspace(GmmParams p, GmmLayout lay, int config, int num_cus);
