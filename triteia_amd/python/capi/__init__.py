from .marlin import mul_2_4, bmm_2_4, sbmm_2_4, sbmm_2_4_multilaunch
from .marlin import sbmm_2_4_routed, sbmm_2_4_planned, route_plan, routed_workspace, pack_2_4
from .punica import add_lora_sgmv_cutlass, add_lora_bgmv, sgmv_routed, lora_scratch, lora_shrink, lora_expand

__all__ = ["mul_2_4", "bmm_2_4", "sbmm_2_4", "sbmm_2_4_multilaunch", "add_lora_sgmv_cutlass", "add_lora_bgmv",
           "sbmm_2_4_routed", "sbmm_2_4_planned", "route_plan", "routed_workspace", "sgmv_routed", "pack_2_4", "lora_scratch", "lora_shrink",
           "lora_expand"]
