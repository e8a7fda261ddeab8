// GENERATED by mlopamd/ops/gen_gemm_w4.py -- do not edit by hand.
// The K-loop of gemm_w4_kernel (csrc/gemm_w4.hip): see the generator's docstring.
#pragma once

#define MLOP_W4_KLOOP_S32_P0_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(48)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_KLOOP_S16_P0_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(32)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_KLOOP_S34_P0_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(50)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_KLOOP_S18_P0_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(34)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "buffer_load_dwordx4 %[vo15], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(16)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "ds_read_b128 %[fa0_7], %[rA0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "ds_read_b128 %[fa1_7], %[rA1] offset:14336\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb0_0], %[fa0_7], a[224:227]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[224:227], %[fb1_0], %[fa1_7], a[224:227]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb0_1], %[fa0_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[228:231], %[fb1_1], %[fa1_7], a[228:231]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb0_2], %[fa0_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[232:235], %[fb1_2], %[fa1_7], a[232:235]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb0_3], %[fa0_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[236:239], %[fb1_3], %[fa1_7], a[236:239]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb0_4], %[fa0_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[240:243], %[fb1_4], %[fa1_7], a[240:243]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb0_5], %[fa0_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[244:247], %[fb1_5], %[fa1_7], a[244:247]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb0_6], %[fa0_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[248:251], %[fb1_6], %[fa1_7], a[248:251]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb0_7], %[fa0_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[252:255], %[fb1_7], %[fa1_7], a[252:255]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn15], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4H_KLOOP_S16_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(28)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4H_KLOOP_S8_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(20)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4H_KLOOP_S18_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(30)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4H_KLOOP_S10_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(22)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(12)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_160_KLOOP_S20_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(33)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_160_KLOOP_S10_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(23)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_160_KLOOP_S22_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(35)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_160_KLOOP_S12_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(25)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(13)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_192_KLOOP_S24_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(38)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_192_KLOOP_S12_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(26)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_192_KLOOP_S26_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(40)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_192_KLOOP_S14_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(28)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(14)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "s_waitcnt lgkmcnt(14)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_224_KLOOP_S28_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(43)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_224_KLOOP_S14_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(29)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_224_KLOOP_S30_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(45)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_224_KLOOP_S16_ASM \
  "s_nop 4\n" \
  "s_mov_b32 %[m0save], m0\n" \
  "s_cmp_eq_u32 %[first], 0\n" \
  "s_cbranch_scc1 L_w4_pref_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[k1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[k1] offen lds\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_branch L_w4_go_%=\n" \
  "L_w4_pref_%=:\n" \
  "s_waitcnt vmcnt(31)\n" \
  "L_w4_go_%=:\n" \
  "s_barrier\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], 0\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], 0\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], 0\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], 0\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], 0\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], 0\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], 0\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], 0\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], 0\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], 0\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], 0\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], 0\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], 0\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cmp_eq_u32 %[iter], 0\n" \
  "s_cbranch_scc1 L_w4_after_%=\n" \
  "L_w4_loop_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "s_barrier\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "buffer_load_dwordx4 %[vo0], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "buffer_load_dwordx4 %[vo1], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "buffer_load_dwordx4 %[vo2], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "buffer_load_dwordx4 %[vo3], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "buffer_load_dwordx4 %[vo4], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "buffer_load_dwordx4 %[vo5], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "buffer_load_dwordx4 %[vo6], %[srdA], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "buffer_load_dwordx4 %[vo7], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "buffer_load_dwordx4 %[vo8], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "buffer_load_dwordx4 %[vo9], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "buffer_load_dwordx4 %[vo10], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "buffer_load_dwordx4 %[vo11], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "buffer_load_dwordx4 %[vo12], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "buffer_load_dwordx4 %[vo13], %[srdB], %[koff] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "buffer_load_dwordx4 %[vo14], %[srdB], %[koff] offen lds\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "s_add_u32 %[koff], %[koff], 0x80\n" \
  "s_cmp_eq_u32 %[koff], %[kend]\n" \
  "s_cselect_b32 %[koff], 0, %[koff]\n" \
  "s_xor_b32 %[dbase], %[dbase], 0x10000\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(15)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "s_sub_u32 %[iter], %[iter], 1\n" \
  "s_cmp_lg_u32 %[iter], 0\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_cbranch_scc1 L_w4_loop_%=\n" \
  "L_w4_after_%=:\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "s_waitcnt vmcnt(0)\n" \
  "s_barrier\n" \
  "v_xor_b32_e32 %[rA0], 0x10000, %[rA0]\n" \
  "v_xor_b32_e32 %[rB0], 0x10000, %[rB0]\n" \
  "v_xor_b32_e32 %[rA1], 0x10000, %[rA1]\n" \
  "v_xor_b32_e32 %[rB1], 0x10000, %[rB1]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "ds_read_b128 %[fa0_0], %[rA0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "ds_read_b128 %[fa1_0], %[rA1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "ds_read_b128 %[fa0_1], %[rA0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "ds_read_b128 %[fb0_0], %[rB0] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "ds_read_b128 %[fb1_0], %[rB1] offset:0\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "ds_read_b128 %[fa1_1], %[rA1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "ds_read_b128 %[fb0_1], %[rB0] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "ds_read_b128 %[fb1_1], %[rB1] offset:2048\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "ds_read_b128 %[fb0_2], %[rB0] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "ds_read_b128 %[fb1_2], %[rB1] offset:4096\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "ds_read_b128 %[fb0_3], %[rB0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "ds_read_b128 %[fb1_3], %[rB1] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "ds_read_b128 %[fb0_4], %[rB0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "ds_read_b128 %[fb1_4], %[rB1] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "ds_read_b128 %[fb0_5], %[rB0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "ds_read_b128 %[fb1_5], %[rB1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb0_0], %[fa0_0], a[0:3]\n" \
  "ds_read_b128 %[fa0_2], %[rA0] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[0:3], %[fb1_0], %[fa1_0], a[0:3]\n" \
  "ds_read_b128 %[fb0_6], %[rB0] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb0_0], %[fa0_1], a[32:35]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[32:35], %[fb1_0], %[fa1_1], a[32:35]\n" \
  "ds_read_b128 %[fb1_6], %[rB1] offset:12288\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb0_1], %[fa0_1], a[36:39]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[36:39], %[fb1_1], %[fa1_1], a[36:39]\n" \
  "ds_read_b128 %[fb0_7], %[rB0] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb0_1], %[fa0_0], a[4:7]\n" \
  "ds_read_b128 %[fb1_7], %[rB1] offset:14336\n" \
  "v_mfma_f32_16x16x32_bf16 a[4:7], %[fb1_1], %[fa1_0], a[4:7]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb0_2], %[fa0_0], a[8:11]\n" \
  "ds_read_b128 %[fa1_2], %[rA1] offset:4096\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[8:11], %[fb1_2], %[fa1_0], a[8:11]\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb0_2], %[fa0_1], a[40:43]\n" \
  "ds_read_b128 %[fa0_3], %[rA0] offset:6144\n" \
  "v_mfma_f32_16x16x32_bf16 a[40:43], %[fb1_2], %[fa1_1], a[40:43]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb0_3], %[fa0_1], a[44:47]\n" \
  "ds_read_b128 %[fa1_3], %[rA1] offset:6144\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[44:47], %[fb1_3], %[fa1_1], a[44:47]\n" \
  "ds_read_b128 %[fa0_4], %[rA0] offset:8192\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb0_3], %[fa0_0], a[12:15]\n" \
  "v_mfma_f32_16x16x32_bf16 a[12:15], %[fb1_3], %[fa1_0], a[12:15]\n" \
  "ds_read_b128 %[fa1_4], %[rA1] offset:8192\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb0_4], %[fa0_0], a[16:19]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[16:19], %[fb1_4], %[fa1_0], a[16:19]\n" \
  "ds_read_b128 %[fa0_5], %[rA0] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb0_4], %[fa0_1], a[48:51]\n" \
  "ds_read_b128 %[fa1_5], %[rA1] offset:10240\n" \
  "v_mfma_f32_16x16x32_bf16 a[48:51], %[fb1_4], %[fa1_1], a[48:51]\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb0_5], %[fa0_1], a[52:55]\n" \
  "ds_read_b128 %[fa0_6], %[rA0] offset:12288\n" \
  "s_waitcnt lgkmcnt(13)\n" \
  "v_mfma_f32_16x16x32_bf16 a[52:55], %[fb1_5], %[fa1_1], a[52:55]\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb0_5], %[fa0_0], a[20:23]\n" \
  "ds_read_b128 %[fa1_6], %[rA1] offset:12288\n" \
  "v_mfma_f32_16x16x32_bf16 a[20:23], %[fb1_5], %[fa1_0], a[20:23]\n" \
  "s_waitcnt lgkmcnt(12)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb0_6], %[fa0_0], a[24:27]\n" \
  "s_waitcnt lgkmcnt(11)\n" \
  "v_mfma_f32_16x16x32_bf16 a[24:27], %[fb1_6], %[fa1_0], a[24:27]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb0_6], %[fa0_1], a[56:59]\n" \
  "v_mfma_f32_16x16x32_bf16 a[56:59], %[fb1_6], %[fa1_1], a[56:59]\n" \
  "s_waitcnt lgkmcnt(10)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb0_7], %[fa0_1], a[60:63]\n" \
  "s_waitcnt lgkmcnt(9)\n" \
  "v_mfma_f32_16x16x32_bf16 a[60:63], %[fb1_7], %[fa1_1], a[60:63]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb0_7], %[fa0_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[28:31], %[fb1_7], %[fa1_0], a[28:31]\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb0_7], %[fa0_2], a[92:95]\n" \
  "s_waitcnt lgkmcnt(8)\n" \
  "v_mfma_f32_16x16x32_bf16 a[92:95], %[fb1_7], %[fa1_2], a[92:95]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb0_6], %[fa0_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[88:91], %[fb1_6], %[fa1_2], a[88:91]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb0_5], %[fa0_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[84:87], %[fb1_5], %[fa1_2], a[84:87]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb0_4], %[fa0_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[80:83], %[fb1_4], %[fa1_2], a[80:83]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb0_3], %[fa0_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[76:79], %[fb1_3], %[fa1_2], a[76:79]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb0_2], %[fa0_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[72:75], %[fb1_2], %[fa1_2], a[72:75]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb0_1], %[fa0_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[68:71], %[fb1_1], %[fa1_2], a[68:71]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb0_0], %[fa0_2], a[64:67]\n" \
  "v_mfma_f32_16x16x32_bf16 a[64:67], %[fb1_0], %[fa1_2], a[64:67]\n" \
  "s_waitcnt lgkmcnt(7)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb0_0], %[fa0_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(6)\n" \
  "v_mfma_f32_16x16x32_bf16 a[96:99], %[fb1_0], %[fa1_3], a[96:99]\n" \
  "s_waitcnt lgkmcnt(5)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb0_0], %[fa0_4], a[128:131]\n" \
  "s_waitcnt lgkmcnt(4)\n" \
  "v_mfma_f32_16x16x32_bf16 a[128:131], %[fb1_0], %[fa1_4], a[128:131]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb0_1], %[fa0_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[132:135], %[fb1_1], %[fa1_4], a[132:135]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb0_1], %[fa0_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[100:103], %[fb1_1], %[fa1_3], a[100:103]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb0_2], %[fa0_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[104:107], %[fb1_2], %[fa1_3], a[104:107]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb0_2], %[fa0_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[136:139], %[fb1_2], %[fa1_4], a[136:139]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb0_3], %[fa0_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[140:143], %[fb1_3], %[fa1_4], a[140:143]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb0_3], %[fa0_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[108:111], %[fb1_3], %[fa1_3], a[108:111]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb0_4], %[fa0_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[112:115], %[fb1_4], %[fa1_3], a[112:115]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb0_4], %[fa0_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[144:147], %[fb1_4], %[fa1_4], a[144:147]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb0_5], %[fa0_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[148:151], %[fb1_5], %[fa1_4], a[148:151]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb0_5], %[fa0_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[116:119], %[fb1_5], %[fa1_3], a[116:119]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb0_6], %[fa0_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[120:123], %[fb1_6], %[fa1_3], a[120:123]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb0_6], %[fa0_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[152:155], %[fb1_6], %[fa1_4], a[152:155]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb0_7], %[fa0_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[156:159], %[fb1_7], %[fa1_4], a[156:159]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb0_7], %[fa0_3], a[124:127]\n" \
  "v_mfma_f32_16x16x32_bf16 a[124:127], %[fb1_7], %[fa1_3], a[124:127]\n" \
  "s_waitcnt lgkmcnt(3)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb0_0], %[fa0_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(2)\n" \
  "v_mfma_f32_16x16x32_bf16 a[160:163], %[fb1_0], %[fa1_5], a[160:163]\n" \
  "s_waitcnt lgkmcnt(1)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb0_0], %[fa0_6], a[192:195]\n" \
  "s_waitcnt lgkmcnt(0)\n" \
  "v_mfma_f32_16x16x32_bf16 a[192:195], %[fb1_0], %[fa1_6], a[192:195]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb0_1], %[fa0_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[196:199], %[fb1_1], %[fa1_6], a[196:199]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb0_1], %[fa0_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[164:167], %[fb1_1], %[fa1_5], a[164:167]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb0_2], %[fa0_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[168:171], %[fb1_2], %[fa1_5], a[168:171]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb0_2], %[fa0_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[200:203], %[fb1_2], %[fa1_6], a[200:203]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb0_3], %[fa0_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[204:207], %[fb1_3], %[fa1_6], a[204:207]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb0_3], %[fa0_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[172:175], %[fb1_3], %[fa1_5], a[172:175]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb0_4], %[fa0_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[176:179], %[fb1_4], %[fa1_5], a[176:179]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb0_4], %[fa0_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[208:211], %[fb1_4], %[fa1_6], a[208:211]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb0_5], %[fa0_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[212:215], %[fb1_5], %[fa1_6], a[212:215]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb0_5], %[fa0_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[180:183], %[fb1_5], %[fa1_5], a[180:183]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb0_6], %[fa0_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[184:187], %[fb1_6], %[fa1_5], a[184:187]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb0_6], %[fa0_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[216:219], %[fb1_6], %[fa1_6], a[216:219]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb0_7], %[fa0_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[220:223], %[fb1_7], %[fa1_6], a[220:223]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb0_7], %[fa0_5], a[188:191]\n" \
  "v_mfma_f32_16x16x32_bf16 a[188:191], %[fb1_7], %[fa1_5], a[188:191]\n" \
  "s_barrier\n" \
  "s_cmp_eq_u32 %[has_next], 0\n" \
  "s_cbranch_scc1 L_w4_end_%=\n" \
  "s_mov_b32 m0, %[dbase]\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n0] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n0] offen lds\n" \
  "s_xor_b32 m0, %[dbase], 0x10000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn0], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn1], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn2], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn3], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn4], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn5], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn6], %[srdA], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn7], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn8], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn9], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn10], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn11], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn12], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn13], %[srdB], %[n1] offen lds\n" \
  "s_add_u32 m0, m0, 0x1000\n" \
  "s_nop 0\n" \
  "buffer_load_dwordx4 %[vn14], %[srdB], %[n1] offen lds\n" \
  "L_w4_end_%=:\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_nop 7\n" \
  "s_mov_b32 m0, %[m0save]\n" \
  ""

#define MLOP_W4_READ0_ASM \
  "v_accvgpr_read_b32 %0, a0\n" \
  "v_accvgpr_read_b32 %1, a1\n" \
  "v_accvgpr_read_b32 %2, a2\n" \
  "v_accvgpr_read_b32 %3, a3\n" \
  "v_accvgpr_read_b32 %4, a4\n" \
  "v_accvgpr_read_b32 %5, a5\n" \
  "v_accvgpr_read_b32 %6, a6\n" \
  "v_accvgpr_read_b32 %7, a7\n" \
  "v_accvgpr_read_b32 %8, a8\n" \
  "v_accvgpr_read_b32 %9, a9\n" \
  "v_accvgpr_read_b32 %10, a10\n" \
  "v_accvgpr_read_b32 %11, a11\n" \
  "v_accvgpr_read_b32 %12, a12\n" \
  "v_accvgpr_read_b32 %13, a13\n" \
  "v_accvgpr_read_b32 %14, a14\n" \
  "v_accvgpr_read_b32 %15, a15\n" \
  "v_accvgpr_read_b32 %16, a16\n" \
  "v_accvgpr_read_b32 %17, a17\n" \
  "v_accvgpr_read_b32 %18, a18\n" \
  "v_accvgpr_read_b32 %19, a19\n" \
  "v_accvgpr_read_b32 %20, a20\n" \
  "v_accvgpr_read_b32 %21, a21\n" \
  "v_accvgpr_read_b32 %22, a22\n" \
  "v_accvgpr_read_b32 %23, a23\n" \
  "v_accvgpr_read_b32 %24, a24\n" \
  "v_accvgpr_read_b32 %25, a25\n" \
  "v_accvgpr_read_b32 %26, a26\n" \
  "v_accvgpr_read_b32 %27, a27\n" \
  "v_accvgpr_read_b32 %28, a28\n" \
  "v_accvgpr_read_b32 %29, a29\n" \
  "v_accvgpr_read_b32 %30, a30\n" \
  "v_accvgpr_read_b32 %31, a31\n" \
  ""

#define MLOP_W4_READ1_ASM \
  "v_accvgpr_read_b32 %0, a32\n" \
  "v_accvgpr_read_b32 %1, a33\n" \
  "v_accvgpr_read_b32 %2, a34\n" \
  "v_accvgpr_read_b32 %3, a35\n" \
  "v_accvgpr_read_b32 %4, a36\n" \
  "v_accvgpr_read_b32 %5, a37\n" \
  "v_accvgpr_read_b32 %6, a38\n" \
  "v_accvgpr_read_b32 %7, a39\n" \
  "v_accvgpr_read_b32 %8, a40\n" \
  "v_accvgpr_read_b32 %9, a41\n" \
  "v_accvgpr_read_b32 %10, a42\n" \
  "v_accvgpr_read_b32 %11, a43\n" \
  "v_accvgpr_read_b32 %12, a44\n" \
  "v_accvgpr_read_b32 %13, a45\n" \
  "v_accvgpr_read_b32 %14, a46\n" \
  "v_accvgpr_read_b32 %15, a47\n" \
  "v_accvgpr_read_b32 %16, a48\n" \
  "v_accvgpr_read_b32 %17, a49\n" \
  "v_accvgpr_read_b32 %18, a50\n" \
  "v_accvgpr_read_b32 %19, a51\n" \
  "v_accvgpr_read_b32 %20, a52\n" \
  "v_accvgpr_read_b32 %21, a53\n" \
  "v_accvgpr_read_b32 %22, a54\n" \
  "v_accvgpr_read_b32 %23, a55\n" \
  "v_accvgpr_read_b32 %24, a56\n" \
  "v_accvgpr_read_b32 %25, a57\n" \
  "v_accvgpr_read_b32 %26, a58\n" \
  "v_accvgpr_read_b32 %27, a59\n" \
  "v_accvgpr_read_b32 %28, a60\n" \
  "v_accvgpr_read_b32 %29, a61\n" \
  "v_accvgpr_read_b32 %30, a62\n" \
  "v_accvgpr_read_b32 %31, a63\n" \
  ""

#define MLOP_W4_READ2_ASM \
  "v_accvgpr_read_b32 %0, a64\n" \
  "v_accvgpr_read_b32 %1, a65\n" \
  "v_accvgpr_read_b32 %2, a66\n" \
  "v_accvgpr_read_b32 %3, a67\n" \
  "v_accvgpr_read_b32 %4, a68\n" \
  "v_accvgpr_read_b32 %5, a69\n" \
  "v_accvgpr_read_b32 %6, a70\n" \
  "v_accvgpr_read_b32 %7, a71\n" \
  "v_accvgpr_read_b32 %8, a72\n" \
  "v_accvgpr_read_b32 %9, a73\n" \
  "v_accvgpr_read_b32 %10, a74\n" \
  "v_accvgpr_read_b32 %11, a75\n" \
  "v_accvgpr_read_b32 %12, a76\n" \
  "v_accvgpr_read_b32 %13, a77\n" \
  "v_accvgpr_read_b32 %14, a78\n" \
  "v_accvgpr_read_b32 %15, a79\n" \
  "v_accvgpr_read_b32 %16, a80\n" \
  "v_accvgpr_read_b32 %17, a81\n" \
  "v_accvgpr_read_b32 %18, a82\n" \
  "v_accvgpr_read_b32 %19, a83\n" \
  "v_accvgpr_read_b32 %20, a84\n" \
  "v_accvgpr_read_b32 %21, a85\n" \
  "v_accvgpr_read_b32 %22, a86\n" \
  "v_accvgpr_read_b32 %23, a87\n" \
  "v_accvgpr_read_b32 %24, a88\n" \
  "v_accvgpr_read_b32 %25, a89\n" \
  "v_accvgpr_read_b32 %26, a90\n" \
  "v_accvgpr_read_b32 %27, a91\n" \
  "v_accvgpr_read_b32 %28, a92\n" \
  "v_accvgpr_read_b32 %29, a93\n" \
  "v_accvgpr_read_b32 %30, a94\n" \
  "v_accvgpr_read_b32 %31, a95\n" \
  ""

#define MLOP_W4_READ3_ASM \
  "v_accvgpr_read_b32 %0, a96\n" \
  "v_accvgpr_read_b32 %1, a97\n" \
  "v_accvgpr_read_b32 %2, a98\n" \
  "v_accvgpr_read_b32 %3, a99\n" \
  "v_accvgpr_read_b32 %4, a100\n" \
  "v_accvgpr_read_b32 %5, a101\n" \
  "v_accvgpr_read_b32 %6, a102\n" \
  "v_accvgpr_read_b32 %7, a103\n" \
  "v_accvgpr_read_b32 %8, a104\n" \
  "v_accvgpr_read_b32 %9, a105\n" \
  "v_accvgpr_read_b32 %10, a106\n" \
  "v_accvgpr_read_b32 %11, a107\n" \
  "v_accvgpr_read_b32 %12, a108\n" \
  "v_accvgpr_read_b32 %13, a109\n" \
  "v_accvgpr_read_b32 %14, a110\n" \
  "v_accvgpr_read_b32 %15, a111\n" \
  "v_accvgpr_read_b32 %16, a112\n" \
  "v_accvgpr_read_b32 %17, a113\n" \
  "v_accvgpr_read_b32 %18, a114\n" \
  "v_accvgpr_read_b32 %19, a115\n" \
  "v_accvgpr_read_b32 %20, a116\n" \
  "v_accvgpr_read_b32 %21, a117\n" \
  "v_accvgpr_read_b32 %22, a118\n" \
  "v_accvgpr_read_b32 %23, a119\n" \
  "v_accvgpr_read_b32 %24, a120\n" \
  "v_accvgpr_read_b32 %25, a121\n" \
  "v_accvgpr_read_b32 %26, a122\n" \
  "v_accvgpr_read_b32 %27, a123\n" \
  "v_accvgpr_read_b32 %28, a124\n" \
  "v_accvgpr_read_b32 %29, a125\n" \
  "v_accvgpr_read_b32 %30, a126\n" \
  "v_accvgpr_read_b32 %31, a127\n" \
  ""

#define MLOP_W4_READ4_ASM \
  "v_accvgpr_read_b32 %0, a128\n" \
  "v_accvgpr_read_b32 %1, a129\n" \
  "v_accvgpr_read_b32 %2, a130\n" \
  "v_accvgpr_read_b32 %3, a131\n" \
  "v_accvgpr_read_b32 %4, a132\n" \
  "v_accvgpr_read_b32 %5, a133\n" \
  "v_accvgpr_read_b32 %6, a134\n" \
  "v_accvgpr_read_b32 %7, a135\n" \
  "v_accvgpr_read_b32 %8, a136\n" \
  "v_accvgpr_read_b32 %9, a137\n" \
  "v_accvgpr_read_b32 %10, a138\n" \
  "v_accvgpr_read_b32 %11, a139\n" \
  "v_accvgpr_read_b32 %12, a140\n" \
  "v_accvgpr_read_b32 %13, a141\n" \
  "v_accvgpr_read_b32 %14, a142\n" \
  "v_accvgpr_read_b32 %15, a143\n" \
  "v_accvgpr_read_b32 %16, a144\n" \
  "v_accvgpr_read_b32 %17, a145\n" \
  "v_accvgpr_read_b32 %18, a146\n" \
  "v_accvgpr_read_b32 %19, a147\n" \
  "v_accvgpr_read_b32 %20, a148\n" \
  "v_accvgpr_read_b32 %21, a149\n" \
  "v_accvgpr_read_b32 %22, a150\n" \
  "v_accvgpr_read_b32 %23, a151\n" \
  "v_accvgpr_read_b32 %24, a152\n" \
  "v_accvgpr_read_b32 %25, a153\n" \
  "v_accvgpr_read_b32 %26, a154\n" \
  "v_accvgpr_read_b32 %27, a155\n" \
  "v_accvgpr_read_b32 %28, a156\n" \
  "v_accvgpr_read_b32 %29, a157\n" \
  "v_accvgpr_read_b32 %30, a158\n" \
  "v_accvgpr_read_b32 %31, a159\n" \
  ""

#define MLOP_W4_READ5_ASM \
  "v_accvgpr_read_b32 %0, a160\n" \
  "v_accvgpr_read_b32 %1, a161\n" \
  "v_accvgpr_read_b32 %2, a162\n" \
  "v_accvgpr_read_b32 %3, a163\n" \
  "v_accvgpr_read_b32 %4, a164\n" \
  "v_accvgpr_read_b32 %5, a165\n" \
  "v_accvgpr_read_b32 %6, a166\n" \
  "v_accvgpr_read_b32 %7, a167\n" \
  "v_accvgpr_read_b32 %8, a168\n" \
  "v_accvgpr_read_b32 %9, a169\n" \
  "v_accvgpr_read_b32 %10, a170\n" \
  "v_accvgpr_read_b32 %11, a171\n" \
  "v_accvgpr_read_b32 %12, a172\n" \
  "v_accvgpr_read_b32 %13, a173\n" \
  "v_accvgpr_read_b32 %14, a174\n" \
  "v_accvgpr_read_b32 %15, a175\n" \
  "v_accvgpr_read_b32 %16, a176\n" \
  "v_accvgpr_read_b32 %17, a177\n" \
  "v_accvgpr_read_b32 %18, a178\n" \
  "v_accvgpr_read_b32 %19, a179\n" \
  "v_accvgpr_read_b32 %20, a180\n" \
  "v_accvgpr_read_b32 %21, a181\n" \
  "v_accvgpr_read_b32 %22, a182\n" \
  "v_accvgpr_read_b32 %23, a183\n" \
  "v_accvgpr_read_b32 %24, a184\n" \
  "v_accvgpr_read_b32 %25, a185\n" \
  "v_accvgpr_read_b32 %26, a186\n" \
  "v_accvgpr_read_b32 %27, a187\n" \
  "v_accvgpr_read_b32 %28, a188\n" \
  "v_accvgpr_read_b32 %29, a189\n" \
  "v_accvgpr_read_b32 %30, a190\n" \
  "v_accvgpr_read_b32 %31, a191\n" \
  ""

#define MLOP_W4_READ6_ASM \
  "v_accvgpr_read_b32 %0, a192\n" \
  "v_accvgpr_read_b32 %1, a193\n" \
  "v_accvgpr_read_b32 %2, a194\n" \
  "v_accvgpr_read_b32 %3, a195\n" \
  "v_accvgpr_read_b32 %4, a196\n" \
  "v_accvgpr_read_b32 %5, a197\n" \
  "v_accvgpr_read_b32 %6, a198\n" \
  "v_accvgpr_read_b32 %7, a199\n" \
  "v_accvgpr_read_b32 %8, a200\n" \
  "v_accvgpr_read_b32 %9, a201\n" \
  "v_accvgpr_read_b32 %10, a202\n" \
  "v_accvgpr_read_b32 %11, a203\n" \
  "v_accvgpr_read_b32 %12, a204\n" \
  "v_accvgpr_read_b32 %13, a205\n" \
  "v_accvgpr_read_b32 %14, a206\n" \
  "v_accvgpr_read_b32 %15, a207\n" \
  "v_accvgpr_read_b32 %16, a208\n" \
  "v_accvgpr_read_b32 %17, a209\n" \
  "v_accvgpr_read_b32 %18, a210\n" \
  "v_accvgpr_read_b32 %19, a211\n" \
  "v_accvgpr_read_b32 %20, a212\n" \
  "v_accvgpr_read_b32 %21, a213\n" \
  "v_accvgpr_read_b32 %22, a214\n" \
  "v_accvgpr_read_b32 %23, a215\n" \
  "v_accvgpr_read_b32 %24, a216\n" \
  "v_accvgpr_read_b32 %25, a217\n" \
  "v_accvgpr_read_b32 %26, a218\n" \
  "v_accvgpr_read_b32 %27, a219\n" \
  "v_accvgpr_read_b32 %28, a220\n" \
  "v_accvgpr_read_b32 %29, a221\n" \
  "v_accvgpr_read_b32 %30, a222\n" \
  "v_accvgpr_read_b32 %31, a223\n" \
  ""

#define MLOP_W4_READ7_ASM \
  "v_accvgpr_read_b32 %0, a224\n" \
  "v_accvgpr_read_b32 %1, a225\n" \
  "v_accvgpr_read_b32 %2, a226\n" \
  "v_accvgpr_read_b32 %3, a227\n" \
  "v_accvgpr_read_b32 %4, a228\n" \
  "v_accvgpr_read_b32 %5, a229\n" \
  "v_accvgpr_read_b32 %6, a230\n" \
  "v_accvgpr_read_b32 %7, a231\n" \
  "v_accvgpr_read_b32 %8, a232\n" \
  "v_accvgpr_read_b32 %9, a233\n" \
  "v_accvgpr_read_b32 %10, a234\n" \
  "v_accvgpr_read_b32 %11, a235\n" \
  "v_accvgpr_read_b32 %12, a236\n" \
  "v_accvgpr_read_b32 %13, a237\n" \
  "v_accvgpr_read_b32 %14, a238\n" \
  "v_accvgpr_read_b32 %15, a239\n" \
  "v_accvgpr_read_b32 %16, a240\n" \
  "v_accvgpr_read_b32 %17, a241\n" \
  "v_accvgpr_read_b32 %18, a242\n" \
  "v_accvgpr_read_b32 %19, a243\n" \
  "v_accvgpr_read_b32 %20, a244\n" \
  "v_accvgpr_read_b32 %21, a245\n" \
  "v_accvgpr_read_b32 %22, a246\n" \
  "v_accvgpr_read_b32 %23, a247\n" \
  "v_accvgpr_read_b32 %24, a248\n" \
  "v_accvgpr_read_b32 %25, a249\n" \
  "v_accvgpr_read_b32 %26, a250\n" \
  "v_accvgpr_read_b32 %27, a251\n" \
  "v_accvgpr_read_b32 %28, a252\n" \
  "v_accvgpr_read_b32 %29, a253\n" \
  "v_accvgpr_read_b32 %30, a254\n" \
  "v_accvgpr_read_b32 %31, a255\n" \
  ""

#define MLOP_W4_128_OPERANDS \
  : [fa0_0] "=&v"(fa0_0), [fa0_1] "=&v"(fa0_1), [fa0_2] "=&v"(fa0_2), [fa0_3] "=&v"(fa0_3), [fa1_0] "=&v"(fa1_0), [fa1_1] "=&v"(fa1_1), \
     [fa1_2] "=&v"(fa1_2), [fa1_3] "=&v"(fa1_3), [fb0_0] "=&v"(fb0_0), [fb0_1] "=&v"(fb0_1), [fb0_2] "=&v"(fb0_2), [fb0_3] "=&v"(fb0_3), \
     [fb0_4] "=&v"(fb0_4), [fb0_5] "=&v"(fb0_5), [fb0_6] "=&v"(fb0_6), [fb0_7] "=&v"(fb0_7), [fb1_0] "=&v"(fb1_0), [fb1_1] "=&v"(fb1_1), \
     [fb1_2] "=&v"(fb1_2), [fb1_3] "=&v"(fb1_3), [fb1_4] "=&v"(fb1_4), [fb1_5] "=&v"(fb1_5), [fb1_6] "=&v"(fb1_6), [fb1_7] "=&v"(fb1_7), \
     [rA0] "+v"(rA0), [rA1] "+v"(rA1), [rB0] "+v"(rB0), [rB1] "+v"(rB1), [koff] "+s"(koff), [dbase] "+s"(dbase), \
     [iter] "+s"(iter), [m0save] "=&s"(m0save) \
  : [vo0] "v"(vo[0]), [vo1] "v"(vo[1]), [vo2] "v"(vo[2]), [vo3] "v"(vo[3]), [vo4] "v"(vo[4]), [vo5] "v"(vo[5]), \
     [vo6] "v"(vo[6]), [vo7] "v"(vo[7]), [vo8] "v"(vo[8]), [vo9] "v"(vo[9]), [vo10] "v"(vo[10]), [vo11] "v"(vo[11]), \
     [vn0] "v"(vn[0]), [vn1] "v"(vn[1]), [vn2] "v"(vn[2]), [vn3] "v"(vn[3]), [vn4] "v"(vn[4]), [vn5] "v"(vn[5]), \
     [vn6] "v"(vn[6]), [vn7] "v"(vn[7]), [vn8] "v"(vn[8]), [vn9] "v"(vn[9]), [vn10] "v"(vn[10]), [vn11] "v"(vn[11]), \
     [srdA] "s"(srdA), [srdB] "s"(srdB), [k0] "s"(k0), [k1] "s"(k1), [n0] "s"(kn0), [n1] "s"(kn1), \
     [kend] "s"(kend), [first] "s"(s_first), [has_next] "s"(s_next) \
  : "memory", "scc", MLOP_W4_AGPR_CLOBBERS

#define MLOP_W4_160_OPERANDS \
  : [fa0_0] "=&v"(fa0_0), [fa0_1] "=&v"(fa0_1), [fa0_2] "=&v"(fa0_2), [fa0_3] "=&v"(fa0_3), [fa0_4] "=&v"(fa0_4), [fa1_0] "=&v"(fa1_0), \
     [fa1_1] "=&v"(fa1_1), [fa1_2] "=&v"(fa1_2), [fa1_3] "=&v"(fa1_3), [fa1_4] "=&v"(fa1_4), [fb0_0] "=&v"(fb0_0), [fb0_1] "=&v"(fb0_1), \
     [fb0_2] "=&v"(fb0_2), [fb0_3] "=&v"(fb0_3), [fb0_4] "=&v"(fb0_4), [fb0_5] "=&v"(fb0_5), [fb0_6] "=&v"(fb0_6), [fb0_7] "=&v"(fb0_7), \
     [fb1_0] "=&v"(fb1_0), [fb1_1] "=&v"(fb1_1), [fb1_2] "=&v"(fb1_2), [fb1_3] "=&v"(fb1_3), [fb1_4] "=&v"(fb1_4), [fb1_5] "=&v"(fb1_5), \
     [fb1_6] "=&v"(fb1_6), [fb1_7] "=&v"(fb1_7), [rA0] "+v"(rA0), [rA1] "+v"(rA1), [rB0] "+v"(rB0), [rB1] "+v"(rB1), \
     [koff] "+s"(koff), [dbase] "+s"(dbase), [iter] "+s"(iter), [m0save] "=&s"(m0save) \
  : [vo0] "v"(vo[0]), [vo1] "v"(vo[1]), [vo2] "v"(vo[2]), [vo3] "v"(vo[3]), [vo4] "v"(vo[4]), [vo5] "v"(vo[5]), \
     [vo6] "v"(vo[6]), [vo7] "v"(vo[7]), [vo8] "v"(vo[8]), [vo9] "v"(vo[9]), [vo10] "v"(vo[10]), [vo11] "v"(vo[11]), \
     [vo12] "v"(vo[12]), [vn0] "v"(vn[0]), [vn1] "v"(vn[1]), [vn2] "v"(vn[2]), [vn3] "v"(vn[3]), [vn4] "v"(vn[4]), \
     [vn5] "v"(vn[5]), [vn6] "v"(vn[6]), [vn7] "v"(vn[7]), [vn8] "v"(vn[8]), [vn9] "v"(vn[9]), [vn10] "v"(vn[10]), \
     [vn11] "v"(vn[11]), [vn12] "v"(vn[12]), [srdA] "s"(srdA), [srdB] "s"(srdB), [k0] "s"(k0), [k1] "s"(k1), \
     [n0] "s"(kn0), [n1] "s"(kn1), [kend] "s"(kend), [first] "s"(s_first), [has_next] "s"(s_next) \
  : "memory", "scc", MLOP_W4_AGPR_CLOBBERS

#define MLOP_W4_192_OPERANDS \
  : [fa0_0] "=&v"(fa0_0), [fa0_1] "=&v"(fa0_1), [fa0_2] "=&v"(fa0_2), [fa0_3] "=&v"(fa0_3), [fa0_4] "=&v"(fa0_4), [fa0_5] "=&v"(fa0_5), \
     [fa1_0] "=&v"(fa1_0), [fa1_1] "=&v"(fa1_1), [fa1_2] "=&v"(fa1_2), [fa1_3] "=&v"(fa1_3), [fa1_4] "=&v"(fa1_4), [fa1_5] "=&v"(fa1_5), \
     [fb0_0] "=&v"(fb0_0), [fb0_1] "=&v"(fb0_1), [fb0_2] "=&v"(fb0_2), [fb0_3] "=&v"(fb0_3), [fb0_4] "=&v"(fb0_4), [fb0_5] "=&v"(fb0_5), \
     [fb0_6] "=&v"(fb0_6), [fb0_7] "=&v"(fb0_7), [fb1_0] "=&v"(fb1_0), [fb1_1] "=&v"(fb1_1), [fb1_2] "=&v"(fb1_2), [fb1_3] "=&v"(fb1_3), \
     [fb1_4] "=&v"(fb1_4), [fb1_5] "=&v"(fb1_5), [fb1_6] "=&v"(fb1_6), [fb1_7] "=&v"(fb1_7), [rA0] "+v"(rA0), [rA1] "+v"(rA1), \
     [rB0] "+v"(rB0), [rB1] "+v"(rB1), [koff] "+s"(koff), [dbase] "+s"(dbase), [iter] "+s"(iter), [m0save] "=&s"(m0save) \
  : [vo0] "v"(vo[0]), [vo1] "v"(vo[1]), [vo2] "v"(vo[2]), [vo3] "v"(vo[3]), [vo4] "v"(vo[4]), [vo5] "v"(vo[5]), \
     [vo6] "v"(vo[6]), [vo7] "v"(vo[7]), [vo8] "v"(vo[8]), [vo9] "v"(vo[9]), [vo10] "v"(vo[10]), [vo11] "v"(vo[11]), \
     [vo12] "v"(vo[12]), [vo13] "v"(vo[13]), [vn0] "v"(vn[0]), [vn1] "v"(vn[1]), [vn2] "v"(vn[2]), [vn3] "v"(vn[3]), \
     [vn4] "v"(vn[4]), [vn5] "v"(vn[5]), [vn6] "v"(vn[6]), [vn7] "v"(vn[7]), [vn8] "v"(vn[8]), [vn9] "v"(vn[9]), \
     [vn10] "v"(vn[10]), [vn11] "v"(vn[11]), [vn12] "v"(vn[12]), [vn13] "v"(vn[13]), [srdA] "s"(srdA), [srdB] "s"(srdB), \
     [k0] "s"(k0), [k1] "s"(k1), [n0] "s"(kn0), [n1] "s"(kn1), [kend] "s"(kend), [first] "s"(s_first), \
     [has_next] "s"(s_next) \
  : "memory", "scc", MLOP_W4_AGPR_CLOBBERS

#define MLOP_W4_224_OPERANDS \
  : [fa0_0] "=&v"(fa0_0), [fa0_1] "=&v"(fa0_1), [fa0_2] "=&v"(fa0_2), [fa0_3] "=&v"(fa0_3), [fa0_4] "=&v"(fa0_4), [fa0_5] "=&v"(fa0_5), \
     [fa0_6] "=&v"(fa0_6), [fa1_0] "=&v"(fa1_0), [fa1_1] "=&v"(fa1_1), [fa1_2] "=&v"(fa1_2), [fa1_3] "=&v"(fa1_3), [fa1_4] "=&v"(fa1_4), \
     [fa1_5] "=&v"(fa1_5), [fa1_6] "=&v"(fa1_6), [fb0_0] "=&v"(fb0_0), [fb0_1] "=&v"(fb0_1), [fb0_2] "=&v"(fb0_2), [fb0_3] "=&v"(fb0_3), \
     [fb0_4] "=&v"(fb0_4), [fb0_5] "=&v"(fb0_5), [fb0_6] "=&v"(fb0_6), [fb0_7] "=&v"(fb0_7), [fb1_0] "=&v"(fb1_0), [fb1_1] "=&v"(fb1_1), \
     [fb1_2] "=&v"(fb1_2), [fb1_3] "=&v"(fb1_3), [fb1_4] "=&v"(fb1_4), [fb1_5] "=&v"(fb1_5), [fb1_6] "=&v"(fb1_6), [fb1_7] "=&v"(fb1_7), \
     [rA0] "+v"(rA0), [rA1] "+v"(rA1), [rB0] "+v"(rB0), [rB1] "+v"(rB1), [koff] "+s"(koff), [dbase] "+s"(dbase), \
     [iter] "+s"(iter), [m0save] "=&s"(m0save) \
  : [vo0] "v"(vo[0]), [vo1] "v"(vo[1]), [vo2] "v"(vo[2]), [vo3] "v"(vo[3]), [vo4] "v"(vo[4]), [vo5] "v"(vo[5]), \
     [vo6] "v"(vo[6]), [vo7] "v"(vo[7]), [vo8] "v"(vo[8]), [vo9] "v"(vo[9]), [vo10] "v"(vo[10]), [vo11] "v"(vo[11]), \
     [vo12] "v"(vo[12]), [vo13] "v"(vo[13]), [vo14] "v"(vo[14]), [vn0] "v"(vn[0]), [vn1] "v"(vn[1]), [vn2] "v"(vn[2]), \
     [vn3] "v"(vn[3]), [vn4] "v"(vn[4]), [vn5] "v"(vn[5]), [vn6] "v"(vn[6]), [vn7] "v"(vn[7]), [vn8] "v"(vn[8]), \
     [vn9] "v"(vn[9]), [vn10] "v"(vn[10]), [vn11] "v"(vn[11]), [vn12] "v"(vn[12]), [vn13] "v"(vn[13]), [vn14] "v"(vn[14]), \
     [srdA] "s"(srdA), [srdB] "s"(srdB), [k0] "s"(k0), [k1] "s"(k1), [n0] "s"(kn0), [n1] "s"(kn1), \
     [kend] "s"(kend), [first] "s"(s_first), [has_next] "s"(s_next) \
  : "memory", "scc", MLOP_W4_AGPR_CLOBBERS

#define MLOP_W4_256_OPERANDS \
  : [fa0_0] "=&v"(fa0_0), [fa0_1] "=&v"(fa0_1), [fa0_2] "=&v"(fa0_2), [fa0_3] "=&v"(fa0_3), [fa0_4] "=&v"(fa0_4), [fa0_5] "=&v"(fa0_5), \
     [fa0_6] "=&v"(fa0_6), [fa0_7] "=&v"(fa0_7), [fa1_0] "=&v"(fa1_0), [fa1_1] "=&v"(fa1_1), [fa1_2] "=&v"(fa1_2), [fa1_3] "=&v"(fa1_3), \
     [fa1_4] "=&v"(fa1_4), [fa1_5] "=&v"(fa1_5), [fa1_6] "=&v"(fa1_6), [fa1_7] "=&v"(fa1_7), [fb0_0] "=&v"(fb0_0), [fb0_1] "=&v"(fb0_1), \
     [fb0_2] "=&v"(fb0_2), [fb0_3] "=&v"(fb0_3), [fb0_4] "=&v"(fb0_4), [fb0_5] "=&v"(fb0_5), [fb0_6] "=&v"(fb0_6), [fb0_7] "=&v"(fb0_7), \
     [fb1_0] "=&v"(fb1_0), [fb1_1] "=&v"(fb1_1), [fb1_2] "=&v"(fb1_2), [fb1_3] "=&v"(fb1_3), [fb1_4] "=&v"(fb1_4), [fb1_5] "=&v"(fb1_5), \
     [fb1_6] "=&v"(fb1_6), [fb1_7] "=&v"(fb1_7), [rA0] "+v"(rA0), [rA1] "+v"(rA1), [rB0] "+v"(rB0), [rB1] "+v"(rB1), \
     [koff] "+s"(koff), [dbase] "+s"(dbase), [iter] "+s"(iter), [m0save] "=&s"(m0save) \
  : [vo0] "v"(vo[0]), [vo1] "v"(vo[1]), [vo2] "v"(vo[2]), [vo3] "v"(vo[3]), [vo4] "v"(vo[4]), [vo5] "v"(vo[5]), \
     [vo6] "v"(vo[6]), [vo7] "v"(vo[7]), [vo8] "v"(vo[8]), [vo9] "v"(vo[9]), [vo10] "v"(vo[10]), [vo11] "v"(vo[11]), \
     [vo12] "v"(vo[12]), [vo13] "v"(vo[13]), [vo14] "v"(vo[14]), [vo15] "v"(vo[15]), [vn0] "v"(vn[0]), [vn1] "v"(vn[1]), \
     [vn2] "v"(vn[2]), [vn3] "v"(vn[3]), [vn4] "v"(vn[4]), [vn5] "v"(vn[5]), [vn6] "v"(vn[6]), [vn7] "v"(vn[7]), \
     [vn8] "v"(vn[8]), [vn9] "v"(vn[9]), [vn10] "v"(vn[10]), [vn11] "v"(vn[11]), [vn12] "v"(vn[12]), [vn13] "v"(vn[13]), \
     [vn14] "v"(vn[14]), [vn15] "v"(vn[15]), [srdA] "s"(srdA), [srdB] "s"(srdB), [k0] "s"(k0), [k1] "s"(k1), \
     [n0] "s"(kn0), [n1] "s"(kn1), [kend] "s"(kend), [first] "s"(s_first), [has_next] "s"(s_next) \
  : "memory", "scc", MLOP_W4_AGPR_CLOBBERS

#define MLOP_W4_AGPR_CLOBBERS "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
